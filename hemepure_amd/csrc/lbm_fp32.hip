// lbm_fp32.hip -- the FP32-shifted collide+stream pass for gfx950.
//
// Same pull step as lbm_fp64.hip (gather the pre-collision state the
// reference holds in fOld, apply the boundary delegates, collide, store the
// post-collision row), with the distributions stored and evolved as
//   g_i = f_i - w_i rho0,   rho0 = 1,
// in float.  Shifting removes the O(w_i) constant part, so float keeps ~7
// significant digits of the deviation from rest instead of of f itself.  In
// shifted form
//   rho = rho0 + sum g,  j = sum c g,
//   g_eq_i = w_i (drho + 3 c.j + 4.5 (c.j)^2 / rho - 1.5 |j|^2 / rho),
// the compressible equilibrium of Lattice.h:374-448 minus w_i rho0; the
// delegates (SBB, BFL, Nash, Ladd) are affine with weights summing to one, so
// they apply to g unchanged.  Iolet densities and speeds arrive in double,
// Windkessel flux terms and the output fields are written in double.
//
// A launch advances every member of a table (see Member32): workgroup tile t
// belongs to member wg_member[t]; a single lattice is a table of one.
#include <hip/hip_runtime.h>

#include <cfloat>

#include "../../include/hemepure_amd.h"
#include "d3q19.h"
#include "device_util.h"
#include "lbm_kernels.h"
#include "windkessel.h"

namespace hlb {

namespace {

constexpr float kW0 = 1.0f / 3.0f, kW1 = 1.0f / 18.0f, kW2 = 1.0f / 36.0f;

__device__ __forceinline__ constexpr float wf(int j) { return j == 0 ? kW0 : (j <= 6 ? kW1 : kW2); }

// Shifted moments: drho = sum g, j = sum c g.  The D3Q19 vectors come in
// opposite pairs (k, k + 1) for odd k, so each pair enters drho through
// g_k + g_k+1 and j through +-(g_k - g_k+1); every sum starts from its first
// term (no addition of a zero).
__device__ __forceinline__ void moments32(const float* g, float& drho, float& jx, float& jy, float& jz) {
  float sp[Q / 2], dp[Q / 2];
#pragma unroll
  for (int p = 0; p < Q / 2; ++p) {
    sp[p] = g[2 * p + 1] + g[2 * p + 2];
    dp[p] = g[2 * p + 1] - g[2 * p + 2];
  }
  drho = g[0];
#pragma unroll
  for (int p = 0; p < Q / 2; ++p) drho += sp[p];
  float j[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    bool first = true;
#pragma unroll
    for (int p = 0; p < Q / 2; ++p) {
      const int c = a == 0 ? CX[2 * p + 1] : (a == 1 ? CY[2 * p + 1] : CZ[2 * p + 1]);
      if (c == 0) continue;
      const float t = c > 0 ? dp[p] : -dp[p];
      j[a] = first ? t : j[a] + t;
      first = false;
    }
  }
  jx = j[0];
  jy = j[1];
  jz = j[2];
}

// c_K . j, the nonzero terms only.
template <int K>
__device__ __forceinline__ float cdotf(float jx, float jy, float jz) {
  constexpr int a = CX[K], b = CY[K], c = CZ[K];
  const float x = a > 0 ? jx : -jx, y = b > 0 ? jy : -jy, z = c > 0 ? jz : -jz;
  if constexpr (K == 0) return 0.0f;
  else if constexpr (a != 0 && b != 0) return x + y;
  else if constexpr (a != 0 && c != 0) return x + z;
  else if constexpr (b != 0 && c != 0) return y + z;
  else if constexpr (a != 0) return x;
  else if constexpr (b != 0) return y;
  else return z;
}

// One shifted equilibrium component; inv = 1 / rho, usq15 = 1.5 |j|^2 / rho.
template <int K>
__device__ __forceinline__ float geq_dir(float drho, float inv, float usq15, float jx, float jy, float jz) {
  const float cu = cdotf<K>(jx, jy, jz);
  return wf(K) * (drho + 3.0f * cu + 4.5f * cu * cu * inv - usq15);
}

template <int K = 0>
__device__ __forceinline__ void geq_all(float drho, float inv, float usq15, float jx, float jy, float jz,
                                        float* geq) {
  if constexpr (K < Q) {
    geq[K] = geq_dir<K>(drho, inv, usq15, jx, jy, jz);
    geq_all<K + 1>(drho, inv, usq15, jx, jy, jz, geq);
  }
}

struct Sym3f {
  float xx, yx, yy, zx, zy, zz;
};

// sum_k c_k c_k v_k.  Opposite vectors share c c^T, so each pair enters
// through v_k + v_k+1, and only the nonzero products are summed.
__device__ __forceinline__ Sym3f second_moments32(const float* v) {
  float sp[Q / 2];
#pragma unroll
  for (int p = 0; p < Q / 2; ++p) sp[p] = v[2 * p + 1] + v[2 * p + 2];
  float r[6];
  // (a, b) component pairs in Sym3f order: xx, yx, yy, zx, zy, zz
  constexpr int A[6] = {0, 1, 1, 2, 2, 2}, B[6] = {0, 0, 1, 0, 1, 2};
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    bool first = true;
#pragma unroll
    for (int p = 0; p < Q / 2; ++p) {
      const int k = 2 * p + 1;
      const int ca = A[e] == 0 ? CX[k] : (A[e] == 1 ? CY[k] : CZ[k]);
      const int cb = B[e] == 0 ? CX[k] : (B[e] == 1 ? CY[k] : CZ[k]);
      if (ca * cb == 0) continue;
      const float t = ca * cb > 0 ? sp[p] : -sp[p];
      r[e] = first ? t : r[e] + t;
      first = false;
    }
  }
  return Sym3f{r[0], r[1], r[2], r[3], r[4], r[5]};
}

// Which A plane set the step reads and writes: k = step index counted from
// the first gathered step; k < 0 is the first step after an initial state.
struct Planes {
  const float* in;
  float* out;
  bool first;
};

__device__ __forceinline__ Planes member_planes(const Member32& m, int step) {
  const int k = m.first0 ? step - 1 : step;
  Planes p;
  p.first = k < 0;
  const int c = k < 0 ? m.cur0 : (m.cur0 ^ (k & 1));
  p.in = k < 0 ? m.F : m.A[c];
  p.out = k < 0 ? m.A[m.cur0] : m.A[c ^ 1];
  return p;
}

// The upstream gather (gather_bb): bounce-back values in the place of wall
// and iolet links.
template <int J = 1>
__device__ __forceinline__ void gather_up32(const float* in, int64_t S, const Lane& L, const uint32_t (&own)[2],
                                            float* g) {
  if constexpr (J < Q) {
    g[J] = gather_bb<J>(uplane(in, S, J < INV[J] ? J : INV[J]), (uint32_t)S, L, own);
    gather_up32<J + 1>(in, S, L, own, g);
  }
}

__device__ __forceinline__ void gather_site32(const float* in, int64_t S, const Lane& L, float* g) {
  const uint32_t own[2] = {L.slot, L.slot + (uint32_t)S};
  g[0] = ldp(in, L.slot);
  gather_up32(in, S, L, own, g);
}

// The boundary delegates of one gathered site, as boundary_fixup in the FP64
// pass (SimpleBounceBackDelegate.h:36-44, BouzidiFirdaousLallemandDelegate.h:
// 44-93).  INNER: the lattice may have links between fluid sites (kInnerLinks).
template <bool INNER>
__device__ __forceinline__ void boundary_fixup32(const Member32& m, const float* in, uint32_t d, uint32_t b,
                                                 const Bnd& r, float* g) {
  float q[Q], own[Q];
  if ((r.far | r.near) != 0) {
#pragma unroll
    for (int k = 1; k < Q; ++k) q[k] = ldp(m.bq + (int64_t)(k - 1) * m.SB, b);
    if (r.far != 0) {
#pragma unroll
      for (int j = 1; j < Q; ++j) own[j] = ldp(uplane(in, m.S, j), d);
      if constexpr (INNER) {
        if (r.far & kInnerLinks) {
          const uint32_t links = ldp(m.gz.inner, b);
#pragma unroll
          for (int j = 1; j < Q; ++j)
            if (links & (1u << (INV[j] - 1))) g[j] = own[INV[j]];
        }
      }
    }
  }
  const uint32_t aside = r.far & r.iolet;
  if (aside != 0) {
#pragma unroll
    for (int j = 1; j < Q; ++j)
      if (aside & (1u << (INV[j] - 1))) g[j] = ldp(plane(m.G, m.SI, j), r.ii);
  }
  if (m.gz.bgz != nullptr && r.wall) {
    const uint32_t gzm = ldp(m.gz.bgz, b);
    const int32_t gzb = ldp(m.gz.bgzbase, b);
#pragma unroll
    for (int j = 1; j < Q; ++j) {
      const uint32_t bit = 1u << (INV[j] - 1);
      if (gzm & bit) g[j] = ldp(m.GW, (uint32_t)(gzb + __builtin_popcount(gzm & (bit - 1u))));
    }
  }
  if ((r.far | r.near) != 0) {
#pragma unroll
    for (int j = 1; j < Q; ++j) {
      const int ib = INV[j];
      const float q2 = 2.0f * q[ib];
      if (r.near & (1u << (j - 1))) g[j] = q2 * g[j] + (1.0f - q2) * g[ib];
      if (r.far & (1u << (j - 1))) g[j] = (g[j] + (q2 - 1.0f) * own[j]) / q2;
    }
  }
}

// What the Nash delegates of a site read per iolet, loaded ahead of the
// collision: ghost density, its deviation, the normal, the Windkessel link.
struct IoletIn32 {
  float rho, drho, n[3];
  uint32_t wk;
};
__device__ __forceinline__ IoletIn32 load_iolet32(const Member32& m, int step, uint32_t gi) {
  const double dens = ldp(m.io_dens + (int64_t)step * m.row, gi);
  return IoletIn32{(float)dens,
                   (float)(dens - 1.0),
                   {ldp(m.io_nf, 3u * gi), ldp(m.io_nf, 3u * gi + 1), ldp(m.io_nf, 3u * gi + 2)},
                   ldp(m.wk_bit, gi)};
}

template <int D = 1>
__device__ __forceinline__ void nash_links32(const Member32& m, float* out, uint32_t slot, const Bnd& r, float drg,
                                             float inv, float usq15, float gx, float gy, float gz) {
  if constexpr (D < Q) {
    if (r.iolet & (1u << (D - 1)))
      stp(iolet_place(D, uplane(out, m.S, D), slot, m.G, m.SI, r), 0, geq_dir<INV[D]>(drg, inv, usq15, gx, gy, gz));
    nash_links32<D + 1>(m, out, slot, r, drg, inv, usq15, gx, gy, gz);
  }
}

struct LaddIn32 {
  double vmax, vmax2;  // the step's speed factors
  float n[3];
};

template <int D0, int D = D0>
__device__ __forceinline__ void ladd_links32(const Member32& m, float* out, uint32_t slot, const Bnd& r,
                                             const LaddIn32& io, const double* s, const double* s2, float rho,
                                             const float* gpost) {
  if constexpr (D < Q && D < D0 + kLaddGroup) {
    if (r.iolet & (1u << (D - 1))) {
      const float v = (float)(io.vmax * s[D - D0] + io.vmax2 * s2[D - D0]);
      const float wx = io.n[0] * v * rho, wy = io.n[1] * v * rho, wz = io.n[2] * v * rho;
      const float correction = 2.0f * wf(D) * cdotf<D>(wx, wy, wz) * 3.0f;
      stp(iolet_place(D, uplane(out, m.S, D), slot, m.G, m.SI, r), 0, gpost[D] - correction);
    }
    ladd_links32<D0, D + 1>(m, out, slot, r, io, s, s2, rho, gpost);
  }
}

// The profile factors of kLaddGroup links at a time, then their values.
template <int D0 = 1>
__device__ __forceinline__ void ladd_groups32(const Member32& m, float* out, uint32_t slot, const Bnd& r,
                                              const LaddIn32& io, float rho, const float* gpost) {
  if constexpr (D0 < Q) {
    double s[kLaddGroup], s2[kLaddGroup];
#pragma unroll
    for (int e = 0; e < kLaddGroup; ++e) {
      if (!(r.iolet & (1u << (D0 + e - 1)))) continue;
      s[e] = ldp(m.ladd_s + (int64_t)(D0 + e - 1) * m.SI, r.ii);
      s2[e] = ldp(m.ladd_s2 + (int64_t)(D0 + e - 1) * m.SI, r.ii);
    }
    ladd_links32<D0>(m, out, slot, r, io, s, s2, rho, gpost);
    ladd_groups32<D0 + kLaddGroup>(m, out, slot, r, io, rho, gpost);
  }
}

// Nash ghost equilibrium (one per site) / Ladd moving-wall bounce-back for
// each iolet link (NashZerothOrderPressureDelegate.h:36-76,
// LaddIoletDelegate.h:37-86), in shifted form, and the Windkessel coupling
// site's flux term.
__device__ __forceinline__ void iolet_links32(const Member32& m, float* out, uint32_t slot, int step, const Bnd& r,
                                              const IoletIn32& io, float rho, float vx, float vy, float vz,
                                              const float* gpost) {
  if (((int)r.gi < m.n_in ? m.inlet_bc : m.outlet_bc) == HLB_IOLET_NASH) {
    const float component = vx * io.n[0] + vy * io.n[1] + vz * io.n[2];
    const float gx = io.n[0] * component * io.rho, gy = io.n[1] * component * io.rho, gz = io.n[2] * component * io.rho;
    const float inv = 1.0f / io.rho;
    const float usq15 = 1.5f * (gx * gx + gy * gy + gz * gz) * inv;
    nash_links32(m, out, slot, r, io.drho, inv, usq15, gx, gy, gz);
  } else {
    const int64_t row = (int64_t)step * m.row;
    ladd_groups32(m, out, slot, r,
                  LaddIn32{ldp(m.io_vmax + row, r.gi), ldp(m.io_vmax2 + row, r.gi), {io.n[0], io.n[1], io.n[2]}}, rho,
                  gpost);
  }
  if (r.iolet & io.wk) {
    const double c = (double)vx * -ldp(m.io_n, 3u * r.gi) + (double)vy * -ldp(m.io_n, 3u * r.gi + 1) +
                     (double)vz * -ldp(m.io_n, 3u * r.gi + 2);
    stp(m.wk_contrib + (step & 1) * m.wk_stride, (uint32_t)ldp(m.wk_pos, r.ii), c);
  }
}

// Wall shear stress magnitude (Lattice.h:1122-1156) from gpost - g.
__device__ __forceinline__ float wall_shear_stress32(const Member32& m, uint32_t b, float tau, const float* g,
                                                     const float* gpost) {
  float dg[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) dg[j] = gpost[j] - g[j];
  const Sym3f s = second_moments32(dg);
  const float fac = -(tau - 0.5f);
  const float p00 = s.xx * fac, p10 = s.yx * fac, p11 = s.yy * fac;
  const float p20 = s.zx * fac, p21 = s.zy * fac, p22 = s.zz * fac;
  const float n0 = ldp(m.bnrm, b), n1 = ldp(m.bnrm + m.SB, b), n2 = ldp(m.bnrm + 2 * m.SB, b);
  const float sv0 = p00 * n0 + p10 * n1 + p20 * n2;
  const float sv1 = p10 * n0 + p11 * n1 + p21 * n2;
  const float sv2 = p20 * n0 + p21 * n1 + p22 * n2;
  const float sq = sv0 * sv0 + sv1 * sv1 + sv2 * sv2;
  const float nn = sv0 * n0 + sv1 * n1 + sv2 * n2;
  return __builtin_sqrtf(sq - nn * nn);
}

// Non-equilibrium parts gneq = g - geq of the opposite pairs (I, I + 1):
// with cu = c_I . j, geq = w (b +- 3 cu), b = a + h cu^2, where
// a = drho - 1.5 |j|^2 / rho and h = 4.5 / rho; each value rounds once per
// multiply-add.
template <int I = 1>
__device__ __forceinline__ void gneq_pairs(const float* g, float a, float h, float jx, float jy, float jz,
                                           float* gneq) {
  if constexpr (I < Q) {
    static_assert(INV[I] == I + 1, "pairs of opposite vectors");
    const float cu = cdotf<I>(jx, jy, jz);
    const float b = __builtin_fmaf(h * cu, cu, a);
    gneq[I] = __builtin_fmaf(-wf(I), __builtin_fmaf(3.0f, cu, b), g[I]);
    gneq[I + 1] = __builtin_fmaf(-wf(I), __builtin_fmaf(-3.0f, cu, b), g[I + 1]);
    gneq_pairs<I + 2>(g, a, h, jx, jy, jz, gneq);
  }
}

// Moments of one site and the relaxation time its collision used.
struct Collision32 {
  float drho, rho, ux, uy, uz, tau;
};

// The collision of one site in shifted form (LBGK.h, TRT.h, LBGKLES.h with
// LBGKLESSpongeLayer::CalculateTau at LBGKLESSpongeLayer.h:122-148): gpost
// from the assembled g.  Every launch variant calls this one function, so all
// of them produce the same bits.
__device__ __forceinline__ Collision32 collide32(const Member32& m, int step, uint32_t d, const float* g,
                                                 float* gpost) {
  Collision32 c;
  float jx, jy, jz;
  moments32(g, c.drho, jx, jy, jz);
  c.rho = 1.0f + c.drho;
  const float inv = __builtin_amdgcn_rcpf(c.rho);
  c.ux = jx * inv;
  c.uy = jy * inv;
  c.uz = jz * inv;
  const float usq15 = 1.5f * __builtin_fmaf(jz, jz, __builtin_fmaf(jy, jy, jx * jx)) * inv;
  const float a = c.drho - usq15;
  float gneq[Q];
  gneq[0] = __builtin_fmaf(-kW0, a, g[0]);
  gneq_pairs(g, a, 4.5f * inv, jx, jy, jz, gneq);
  c.tau = m.tau;
  if (m.kernel == HLB_KERNEL_TRT) {
    gpost[0] = __builtin_fmaf(m.omega, gneq[0], g[0]);
#pragma unroll
    for (int i = 1; i < Q; i += 2) {
      const float sum = gneq[i] + gneq[i + 1], dif = gneq[i] - gneq[i + 1];
      gpost[i] = __builtin_fmaf(m.half_omega_minus, dif, __builtin_fmaf(m.half_omega, sum, g[i]));
      gpost[i + 1] = __builtin_fmaf(-m.half_omega_minus, dif, __builtin_fmaf(m.half_omega, sum, g[i + 1]));
    }
    return c;
  }
  float om = m.omega;
  if (m.kernel == HLB_KERNEL_LES) {
    const Sym3f q = second_moments32(gneq);
    const float off = __builtin_fmaf(q.zy, q.zy, __builtin_fmaf(q.zx, q.zx, q.yx * q.yx));
    const float q2 = __builtin_fmaf(2.0f, off, __builtin_fmaf(q.zz, q.zz, __builtin_fmaf(q.yy, q.yy, q.xx * q.xx)));
    const float root = __builtin_amdgcn_sqrtf(__builtin_fmaf(m.les_k, __builtin_amdgcn_sqrtf(q2), m.tau * m.tau));
    c.tau = 0.5f * (m.tau + root);
    if (m.vtau != nullptr) {
      const double t = ldp(m.sp_t + (int64_t)step * m.row, 0);
      if (t >= 0.0) {
        const float vt = ldp(m.vtau, d);
        if (t <= m.sp_half) c.tau = vt == m.tau ? c.tau : vt;
        else c.tau = (c.tau - vt) * 2.0f / (float)m.sp_life * (float)t + (2.0f * vt - c.tau);
      }
    }
    om = -__builtin_amdgcn_rcpf(c.tau);
  }
#pragma unroll
  for (int j = 0; j < Q; ++j) gpost[j] = __builtin_fmaf(gneq[j], om, g[j]);
  return c;
}

// The post-collision row of a site: 19 stores, non-temporal ones for NT.
template <bool NT>
__device__ __forceinline__ void store_row32(const Member32& m, float* out, uint32_t d, const float* gpost) {
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    if constexpr (NT) stp_nt(uplane(out, m.S, j), d, gpost[j]);
    else stp(uplane(out, m.S, j), d, gpost[j]);
  }
}

// The member of a tile, made wave-uniform so the record is read with scalar
// loads.
__device__ __forceinline__ int member_of_tile(const int32_t* wg_member, uint32_t tile) {
  return wg_member ? __builtin_amdgcn_readfirstlane(ldp(wg_member, tile)) : 0;
}

// One site of a slab in flight: its lane, boundary record and the
// pre-collision g being assembled.
struct Site32 {
  Lane L;
  bool ok;
  Bnd bnd;
  float g[Q];
};

// Decodes slab record r for this lane and issues the site's gathers (the
// loads are not waited for here).
__device__ __forceinline__ void site_gather32(const Member32& m, const Planes& P, uint32_t r, Site32& s) {
  s.bnd = no_bnd();
  s.ok = slab_lane(m.bt, r, s.L);
  if (!s.ok) return;
  if (s.L.boundary) s.bnd = load_bnd(m.bnd, s.L.b);
  if (P.first) {
#pragma unroll
    for (int j = 0; j < Q; ++j) s.g[j] = ldp(uplane(P.in, m.S, j), s.L.slot);
  } else {
    gather_site32(P.in, m.S, s.L, s.g);
  }
}

// The boundary delegates, the GZS staging, collision, stores, iolet values
// and property fields of one gathered site.
template <bool NT>
__device__ __forceinline__ void site_finish32(const Member32& m, const Planes& P, int step, const Lane& L, const Bnd& bnd,
                                              const float* g) {
  const uint32_t d = L.slot;
  IoletIn32 io{};
  if (bnd.iolet != 0) io = load_iolet32(m, step, bnd.gi);
  if (m.gz.pmask != nullptr) {
    const uint64_t pm = uniform64(ldp(m.gz.pmask, L.r));
    if ((pm >> (threadIdx.x & 63u)) & 1u) {
      const uint32_t pi = (uint32_t)__builtin_amdgcn_readfirstlane(ldp(m.gz.pbase, L.r)) + lanes_below(pm);
#pragma unroll
      for (int j = 0; j < Q; ++j) stp(plane(m.P, m.gz.SP, j), pi, g[j]);
    }
  }

  float gpost[Q];
  const Collision32 cs = collide32(m, step, d, g, gpost);
  store_row32<NT>(m, P.out, d, gpost);

  if (bnd.iolet != 0) iolet_links32(m, P.out, d, step, bnd, io, cs.rho, cs.ux, cs.uy, cs.uz, gpost);
  if (step == m.props_at) {
    stp(m.rho, d, 1.0 + (double)cs.drho);
    stp(m.u, d, (double)cs.ux);
    stp(plane(m.u, m.S, 1), d, (double)cs.uy);
    stp(plane(m.u, m.S, 2), d, (double)cs.uz);
    const float w = bnd.wall ? wall_shear_stress32(m, L.b, cs.tau, g, gpost) : FLT_MAX;
    stp(m.wss, d, w == FLT_MAX ? DBL_MAX : (double)w);
  }
}

// B threads per workgroup tile, each wavefront SPT consecutive slabs (the
// gathers of all of them issued before any is waited for); ORDER: the tile
// order (TileOrder); NT: non-temporal stores of the post-collision rows.
template <int B, int ORDER, int W = 0, int SPT = 1, bool NT = false, bool INNER = false>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(W > 0 ? W : 1))) void step_fp32(
    const Member32* __restrict__ members, const int32_t* __restrict__ wg_member, int step, WkLaunch wk) {
  if (wk_workgroup(wk, step)) return;
  const uint32_t tile = tile_index<ORDER>(wk.groups);
  const int mi = member_of_tile(wg_member, tile);
  if (mi < 0) return;  // padding tile
  const Member32& m = members[mi];
  const uint32_t r0 =
      ((tile - m.wg_begin) * (B / kSlab) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * (uint32_t)SPT;
  const Planes P = member_planes(m, step);
  if constexpr (SPT == 1) {
    Lane L;
    if (!slab_lane(m.bt, r0, L)) return;
    Bnd bnd = no_bnd();
    if (L.boundary) bnd = load_bnd(m.bnd, L.b);
    float g[Q];
    if (P.first) {
#pragma unroll
      for (int j = 0; j < Q; ++j) g[j] = ldp(uplane(P.in, m.S, j), L.slot);
    } else {
      gather_site32(P.in, m.S, L, g);
      if (L.boundary) boundary_fixup32<INNER>(m, P.in, L.slot, L.b, bnd, g);
    }
    site_finish32<NT>(m, P, step, L, bnd, g);
  } else {
    Site32 s[SPT];
#pragma unroll
    for (int k = 0; k < SPT; ++k) site_gather32(m, P, r0 + (uint32_t)k, s[k]);
#pragma unroll
    for (int k = 0; k < SPT; ++k) {
      if (!s[k].ok) continue;
      if (!P.first && s[k].L.boundary) boundary_fixup32<INNER>(m, P.in, s[k].L.slot, s[k].L.b, s[k].bnd, s[k].g);
      site_finish32<NT>(m, P, step, s[k].L, s[k].bnd, s[k].g);
    }
  }
}

// Guo-Zheng-Shi links in the shifted form (see gzs_links_fp64): the wall
// node keeps this site's density, so its shifted equilibrium uses the same
// drho.
__global__ __launch_bounds__(kBlock) void gzs_links_fp32(const Member32* __restrict__ members,
                                                         const GzsLink* __restrict__ links, int n, int step) {
  const int e = blockIdx.x * kBlock + threadIdx.x;
  if (e >= n) return;
  const Member32& m = members[0];
  const GzsLink lk = links[e];
  const int d = lk.dir, i = INV[d];
  const float q = lk.q;
  float g[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) g[j] = ldp(plane(m.P, m.gz.SP, j), (uint32_t)lk.site_p);
  float drho, jx, jy, jz;
  moments32(g, drho, jx, jy, jz);
  const float rho = 1.0f + drho, inv = 1.0f / rho;
  float geq[Q], gneq[Q];
  geq_all(drho, inv, 1.5f * (jx * jx + jy * jy + jz * jz) * inv, jx, jy, jz, geq);
#pragma unroll
  for (int j = 0; j < Q; ++j) gneq[j] = g[j] - geq[j];
  const float fac = 1.0f - 1.0f / q;
  float wj[3] = {jx * fac, jy * fac, jz * fac};
  if (lk.mode == 2) {
    float h[Q];
#pragma unroll
    for (int j = 0; j < Q; ++j) h[j] = ldp(plane(m.P, m.gz.SP, j), (uint32_t)lk.nb_p);
    float hd, hx, hy, hz;
    moments32(h, hd, hx, hy, hz);
    const float hr = 1.0f + hd, hinv = 1.0f / hr;
    float heq[Q];
    geq_all(hd, hinv, 1.5f * (hx * hx + hy * hy + hz * hz) * hinv, hx, hy, hz, heq);
    const float hv[3] = {hx * hinv, hy * hinv, hz * hinv};
#pragma unroll
    for (int c = 0; c < 3; ++c) wj[c] = q * wj[c] + (1.0f - q) * rho * (hv[c] * (q - 1.0f) / (q + 1.0f));
#pragma unroll
    for (int j = 0; j < Q; ++j) gneq[j] = q * gneq[j] + (1.0f - q) * (h[j] - heq[j]);
  } else if (lk.mode == 3) {
    const double* vmax = m.io_vmax + (int64_t)step * m.row;
    const double* vmax2 = m.io_vmax2 + (int64_t)step * m.row;
    const float sp = (float)(ldp(vmax, (uint32_t)lk.gi) * lk.s + ldp(vmax2, (uint32_t)lk.gi) * lk.s2);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const float v = (float)ldp(m.io_n, 3u * lk.gi + c) * sp;
      wj[c] = q * wj[c] + (1.0f - q) * rho * (v * (q - 1.0f) / (q + 1.0f));
    }
  }
  float weq[Q];
  geq_all(drho, inv, 1.5f * (wj[0] * wj[0] + wj[1] * wj[1] + wj[2] * wj[2]) * inv, wj[0], wj[1], wj[2], weq);
  float val;
  if (m.kernel == HLB_KERNEL_TRT) {
    const int lo = i < INV[i] ? i : INV[i], hi = i < INV[i] ? INV[i] : i;
    const float sym = m.half_omega * (gneq[lo] + gneq[hi]);
    const float asym = m.half_omega_minus * (gneq[lo] - gneq[hi]);
    val = i == lo ? weq[lo] + gneq[lo] + sym + asym : weq[hi] + gneq[hi] + sym - asym;
  } else {
    val = weq[i] + gneq[i] + gneq[i] * m.omega;
  }
  stp(const_cast<float*>(m.GW), (uint32_t)e, val);
}

// Pre-collision g entering the next step into F (device order), for
// downloads and the stability scan.
__device__ __forceinline__ uint32_t slab_record4() {
  return xcd_tile() * (kBlock / kSlab) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

__global__ __launch_bounds__(kBlock) void gather_fp32(const Member32* __restrict__ members, float* __restrict__ F) {
  const Member32& m = members[0];
  Lane L;
  if (!slab_lane(m.bt, slab_record4(), L)) return;
  const float* in = m.A[m.cur0];
  Bnd bnd = no_bnd();
  if (L.boundary) bnd = load_bnd(m.bnd, L.b);
  float g[Q];
  gather_site32(in, m.S, L, g);
  if (L.boundary) boundary_fixup32<true>(m, in, L.slot, L.b, bnd, g);
#pragma unroll
  for (int j = 0; j < Q; ++j) stp(plane(F, m.S, j), L.slot, g[j]);
}

__global__ __launch_bounds__(kBlock) void fill_planes_fp32(float* __restrict__ F, int64_t N, int64_t S,
                                                           const float* __restrict__ vals) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k >= N) return;
#pragma unroll
  for (int j = 0; j < Q; ++j) F[(int64_t)j * S + k] = vals[j];
}

// StabilityTester on the shifted storage: f = g + w > 0 at every fluid site.
__global__ __launch_bounds__(kBlock) void unstable_fp32(BrickTables bt, const float* __restrict__ F, int64_t S,
                                                        int* __restrict__ flag) {
  Lane L;
  if (!slab_lane(bt, slab_record4(), L)) return;
  bool bad = false;
#pragma unroll
  for (int j = 0; j < Q; ++j) bad |= !(ldp(plane(F, S, j), L.slot) > -wf(j));
  if (bad) *flag = 1;
}

// Cycle-to-cycle change of the velocity field: max over sites and components
// of |u - prev| (prev is the float snapshot of the previous cycle), then
// prev <- u.  The maximum is combined per wavefront and then across waves with
// an unsigned atomic max on the float bits (exact for non-negative floats).
// A NaN velocity reports +inf.
__global__ __launch_bounds__(kBlock) void cycle_delta(const double* __restrict__ u, float* __restrict__ prev,
                                                      int64_t N, int64_t S, unsigned* __restrict__ out_bits) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  float d = 0.0f;
  if (k < N) {
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const double v = u[(int64_t)a * S + k];
      const float pv = prev[(int64_t)a * S + k];
      const double e = __builtin_fabs(v - (double)pv);
      d = (e == e) ? __builtin_fmaxf(d, (float)e) : __builtin_inff();
      prev[(int64_t)a * S + k] = (float)v;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) d = __builtin_fmaxf(d, __shfl_xor(d, off, 64));
  if ((threadIdx.x & 63) == 0) atomicMax(out_bits, __float_as_uint(d));
}

}  // namespace

hipError_t launch_cycle_delta(const double* u, float* prev, int64_t N, int64_t S, unsigned* out_bits,
                              hipStream_t s) {
  if (N == 0) return hipSuccess;
  hipLaunchKernelGGL(cycle_delta, dim3((unsigned)((N + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, u, prev, N, S,
                     out_bits);
  return hipGetLastError();
}

LaunchShape launch_shape(int variant, bool fp32) {
  static const int kBlocks6[6] = {128, 128, 256, 256, 64, 64}, kBlocks3[3] = {128, 256, 64};
  LaunchShape l{};
  l.spt = 1;
  int u = variant;
  const int base = fp32 ? kFp32Shapes : kFp64Shapes;
  l.nt = u >= base;
  if (l.nt) u -= base;
  bool chunks = false;
  if (fp32) {
    // 0..35 and 36..71: plain / XCD shapes with one and two slabs per
    // wavefront; 72..89 and 90..107: XCD-chunk shapes likewise
    chunks = u >= 2 * kShapeVariants;
    if (chunks) u -= 2 * kShapeVariants;
    const int per = chunks ? kChunkVariants : kShapeVariants;
    if (u >= per) {
      l.spt = 2;
      u -= per;
    }
  } else {
    chunks = u >= kShapeVariants;
    if (chunks) u -= kShapeVariants;
  }
  if (!chunks) {
    l.block = kBlocks6[u % 6];
    l.order = (u % 6) & 1 ? kOrderXcd : kOrderPlain;
    l.level = u / 6;
  } else {
    l.block = kBlocks3[u % 3];
    l.order = kOrderXcdChunks;
    l.level = u / 3;
  }
  return l;
}

unsigned shape_lds(const LaunchShape& l) {
  // 160 KB of LDS per CU, four SIMDs: w waves per SIMD <=> 160 KB / (4 w) per wave.
  static const unsigned per_wave[6] = {0u, 10240u, 13653u, 20480u, 0u, 0u};
  return per_wave[l.level] * (unsigned)(l.block / 64);
}

// `grid` workgroup tiles of the variant's size, padded as shape_grid pads
// them (padding tiles map to member -1).  inner: a member has links between
// fluid sites, and the variant is an inner_launch one.
hipError_t launch_step_fp32(const Member32* members, const int32_t* wg_member, uint32_t grid, int step,
                            const WkLaunch& wk, int variant, bool inner, hipStream_t s) {
  if (grid == 0) return hipSuccess;
  grid += wk.groups;
  const LaunchShape l = launch_shape(variant, true);
  if (inner) {
    if (l.nt)
      hipLaunchKernelGGL((step_fp32<kSlab, kOrderXcd, 0, 1, true, true>), dim3(grid), dim3(kSlab), 0, s, members,
                         wg_member, step, wk);
    else
      hipLaunchKernelGGL((step_fp32<kSlab, kOrderXcd, 0, 1, false, true>), dim3(grid), dim3(kSlab), 0, s, members,
                         wg_member, step, wk);
    return hipGetLastError();
  }
  const unsigned lds = shape_lds(l);
#define HLB_VN(B, O, W, NT)                                                                                  \
  if (l.spt == 2)                                                                                            \
    hipLaunchKernelGGL((step_fp32<B, O, W, 2, NT>), dim3(grid), dim3(B), lds, s, members, wg_member, step, wk);  \
  else                                                                                                       \
    hipLaunchKernelGGL((step_fp32<B, O, W, 1, NT>), dim3(grid), dim3(B), lds, s, members, wg_member, step, wk)
#define HLB_V(B, O, W)     \
  if (l.nt) {              \
    HLB_VN(B, O, W, true); \
  } else {                 \
    HLB_VN(B, O, W, false); \
  }
#define HLB_ORDERS(B, W)                              \
  switch (l.order) {                                  \
    case kOrderPlain: HLB_V(B, kOrderPlain, W); break; \
    case kOrderXcd: HLB_V(B, kOrderXcd, W); break;     \
    default: HLB_V(B, kOrderXcdChunks, W); break;      \
  }
#define HLB_SHAPES(W)                   \
  switch (l.block) {                    \
    case 128: HLB_ORDERS(128, W); break; \
    case 256: HLB_ORDERS(256, W); break; \
    default: HLB_ORDERS(64, W); break;   \
  }
  // the FP32 kernel fits 5 waves per SIMD as compiled; levels 4, 5 ask for 6, 7
  switch (l.level) {
    case 4: HLB_SHAPES(6); break;
    case 5: HLB_SHAPES(7); break;
    default: HLB_SHAPES(0); break;
  }
#undef HLB_SHAPES
#undef HLB_ORDERS
#undef HLB_V
#undef HLB_VN
  return hipGetLastError();
}

static uint32_t slab_grid4(int64_t nslab) {
  const int64_t wg = (nslab + kBlock / kSlab - 1) / (kBlock / kSlab);
  return (uint32_t)((wg + kXcds - 1) / kXcds * kXcds);
}

hipError_t launch_gzs_fp32(const Member32* members, const GzsLink* links, int n, int step, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(gzs_links_fp32, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, members, links, n, step);
  return hipGetLastError();
}

hipError_t launch_gather_fp32(const Member32* members, int64_t nslab, float* F, hipStream_t s) {
  if (nslab == 0) return hipSuccess;
  const uint32_t grid = slab_grid4(nslab);
  hipLaunchKernelGGL(gather_fp32, dim3(grid), dim3(kBlock), 0, s, members, F);
  return hipGetLastError();
}

hipError_t launch_fill_fp32(float* F, int64_t N, int64_t S, const float* vals, hipStream_t s) {
  if (N == 0) return hipSuccess;
  hipLaunchKernelGGL(fill_planes_fp32, dim3((unsigned)((N + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, F, N, S,
                     vals);
  return hipGetLastError();
}

hipError_t launch_unstable_fp32(const BrickTables& bt, const float* F, int64_t S, int* flag, hipStream_t s) {
  if (bt.nslab == 0) return hipSuccess;
  hipLaunchKernelGGL(unstable_fp32, dim3(slab_grid4(bt.nslab)), dim3(kBlock), 0, s, bt, F, S, flag);
  return hipGetLastError();
}

}  // namespace hlb
