// lbm_fp64.hip -- the fused double-precision collide+stream pass for gfx950.
//
// One wavefront per slab (one x layer of an 8^3 brick, 64 lanes = the
// layer's (y, z) positions), slabs in the compact slab layout of
// lbm_kernels.h; a workgroup tile holds one, two or four slabs (the launch
// shape the autotuner picks).  A step of the reference is
//   collide at every site, push fPost[d] to the neighbour (or a boundary
//   delegate writes the site's own slot), BFL post-step, swap
// (src/lb/lb.hpp:192-347).  Here the same step is one pull pass: each site
// first materialises the pre-collision f it would hold in the reference's
// fOld by gathering the previous pass's post-collision values (plain links:
// the neighbour's value; SimpleBounceBack / BFL: the site's own values,
// src/lb/streamers/SimpleBounceBackDelegate.h:36-44,
// BouzidiFirdaousLallemandDelegate.h:44-93; Nash / Ladd: the value its iolet
// delegate computed last pass), then collides and stores its own
// post-collision row.  Neighbour slots come from the slab record's fluid
// masks and bases (device_util.h), not from a table; stores are coalesced
// per plane; the 18 gathers read the same or an adjacent slab.
//
// Tiles can be mapped XCD-contiguously: the hardware hands workgroup w to
// XCD w mod 8, so logical tile (w mod 8) * (grid / 8) + w / 8 gives each
// XCD one contiguous eighth of the slabs, and the lines a tile's
// neighbours also read stay in that XCD's L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cstdlib>

#include "../../include/hemepure_amd.h"
#include "d3q19.h"
#include "device_util.h"
#include "lbm_kernels.h"
#include "windkessel.h"

namespace hlb {

namespace {

// Gathers the pre-collision values, bounce-back ones in the place of wall and
// iolet links.  NARROW: each pair of opposite planes fits 32-bit offsets from
// its lower plane; otherwise the plane is picked with the 64-bit address.
template <bool NARROW, int J = 1>
__device__ __forceinline__ void gather_up(const StepArgs& a, const Lane& L, const uint32_t (&own)[2], double* f) {
  if constexpr (J < Q) {
    if constexpr (NARROW) {
      f[J] = gather_bb<J>(a.ain[J < INV[J] ? J : INV[J]], (uint32_t)a.S, L, own);
    } else {
      uint64_t fluid = 0;
      const uint32_t up = upstream_pos<J>(L, fluid);
      const bool plain = __builtin_amdgcn_inverse_ballot_w64(fluid);
      f[J] = *(const HLB_GLOBAL double*)((plain ? a.ain[J] : a.ain[INV[J]]) + (plain ? up : L.slot));
    }
    gather_up<NARROW, J + 1>(a, L, own, f);
  }
}

template <bool NARROW>
__device__ __forceinline__ void gather_site(const StepArgs& a, const Lane& L, double* f) {
  const uint32_t own[2] = {L.slot, L.slot + (uint32_t)a.S};
  f[0] = ldp(a.ain[0], L.slot);
  gather_up<NARROW>(a, L, own, f);
}

// The boundary delegates of one gathered site: f[j] already holds what the
// site's own slot has in plane INV[j] for every wall or iolet link INV[j]: the
// post-collision value at a wall link, which is all
// SimpleBounceBackDelegate.h:36-44 does, and the iolet delegate's value at an
// iolet link (iolet_links).  Where such a link leads to a fluid site it holds the
// neighbour's value, and the site's own takes its place (kInnerLinks).
//
// A wave with boundary lanes is bound by instructions and by the chain of
// loads it waits for, not by bytes.  So what each direction does is worked out
// on the host (BndRec: one bit test and, where no lane of the wave has it, one
// skipped branch) and all loads are issued before any value is used.  With the
// masks formed from the link masks per direction and the own values loaded
// where they were needed, a wave spent ~800 more vector instructions and up to
// a round of loads per link: the Y-bifurcation (0.70M sites) 46.2 -> 41.7 us a
// step, the 30k-site cylinder, where the iolet layers' waves decide, 9.0 ->
// 6.4 us, FP32: 29.1 -> 27.3 us, the 20-pipe ensemble 78.8 -> 72.9 us.
__device__ __forceinline__ void boundary_fixup(const StepArgs& a, uint32_t d, uint32_t b, const Bnd& r, double* f) {
  float q[Q];
  double own[Q];
  if ((r.far | r.near) != 0) {
#pragma unroll
    for (int k = 1; k < Q; ++k) q[k] = ldp(a.bq + (int64_t)(k - 1) * a.SB, b);
    if (r.far != 0) {
#pragma unroll
      for (int j = 1; j < Q; ++j) own[j] = ldp(a.ain[j], d);
      if (r.far & kInnerLinks) {
        const uint32_t links = ldp(a.gz.inner, b);
#pragma unroll
        for (int j = 1; j < Q; ++j)
          if (links & (1u << (INV[j] - 1))) f[j] = own[INV[j]];
      }
    }
  }
  const uint32_t aside = r.far & r.iolet;
  if (aside != 0) {
#pragma unroll
    for (int j = 1; j < Q; ++j)
      if (aside & (1u << (INV[j] - 1))) f[j] = ldp(plane(a.G, a.SI, j), r.ii);
  }
  if (a.gz.bgz != nullptr && r.wall) {
    // GuoZhengShiDelegate: the link kernel's values.
    const uint32_t gzm = ldp(a.gz.bgz, b);
    const int32_t gzb = ldp(a.gz.bgzbase, b);
#pragma unroll
    for (int j = 1; j < Q; ++j) {
      const uint32_t bit = 1u << (INV[j] - 1);
      if (gzm & bit) f[j] = ldp(a.GW, (uint32_t)(gzb + __builtin_popcount(gzm & (bit - 1u))));
    }
  }
  if ((r.far | r.near) != 0) {
    // BouzidiFirdaousLallemandDelegate.h: the stream of a wall link ib =
    // INV[j] with q >= 1/2 (:44-70) and the post-step of one with q < 1/2
    // (:72-93).  The post-step reads the streamed f[ib], which no other
    // interpolation of the site writes.
#pragma unroll
    for (int j = 1; j < Q; ++j) {
      const int ib = INV[j];
      const double q2 = 2.0 * (double)q[ib];
      if (r.near & (1u << (j - 1))) f[j] = q2 * f[j] + (1.0 - q2) * f[ib];
      if (r.far & (1u << (j - 1))) f[j] = (f[j] + (q2 - 1) * own[j]) / q2;
    }
  }
}

// What the iolet delegates of a site read per iolet, loaded ahead of the
// row's stores: ghost density, normal, the Windkessel link.
struct IoletIn {
  double dens, n[3];
  uint32_t wk;
};
__device__ __forceinline__ IoletIn load_iolet(const StepArgs& a, uint32_t gi) {
  return IoletIn{a.io_dens[gi], {a.io_n[3 * gi], a.io_n[3 * gi + 1], a.io_n[3 * gi + 2]}, a.wk_bit[gi]};
}

template <int D = 1>
__device__ __forceinline__ void nash_links(const StepArgs& a, uint32_t slot, const Bnd& r, const FeqPre& p, double gx,
                                           double gy, double gz) {
  if constexpr (D < Q) {
    if (r.iolet & (1u << (D - 1))) stp(iolet_place(D, a.aout[D], slot, a.G, a.SI, r), 0, feq_dir<INV[D]>(p, gx, gy, gz));
    nash_links<D + 1>(a, slot, r, p, gx, gy, gz);
  }
}

// Iolet delegates of one site, after its row's stores: the value each iolet
// link k hands to the next step in direction INV[k].  Nash: f_eq of the ghost
// state, one per site (NashZerothOrderPressureDelegate.h:36-76; the normal is
// its float copy).  Ladd: bounce-back minus the moving-wall correction
// (LaddIoletDelegate.h:37-86).
__device__ __forceinline__ void iolet_links(const StepArgs& a, uint32_t slot, const Bnd& r, const IoletIn& io, int bc,
                                            double rho, double vx, double vy, double vz, const double* fpost) {
  if (bc == HLB_IOLET_NASH) {
    const double rg = io.dens;
    const double nx = (double)(float)io.n[0], ny = (double)(float)io.n[1], nz = (double)(float)io.n[2];
    const double component = vx * nx + vy * ny + vz * nz;
    const double gx = nx * component * rg, gy = ny * component * rg, gz = nz * component * rg;
    nash_links(a, slot, r, feq_pre(rg, gx, gy, gz), gx, gy, gz);
  } else {
    const double vmax = a.io_vmax[r.gi], vmax2 = a.io_vmax2[r.gi];
#pragma unroll
    for (int d0 = 1; d0 < Q; d0 += kLaddGroup) {
      double s[kLaddGroup], s2[kLaddGroup];
#pragma unroll
      for (int e = 0; e < kLaddGroup; ++e) {
        if (!(r.iolet & (1u << (d0 + e - 1)))) continue;
        s[e] = ldp(a.ladd_s + (int64_t)(d0 + e - 1) * a.SI, r.ii);
        s2[e] = ldp(a.ladd_s2 + (int64_t)(d0 + e - 1) * a.SI, r.ii);
      }
#pragma unroll
      for (int e = 0; e < kLaddGroup; ++e) {
        const int d = d0 + e;
        if (!(r.iolet & (1u << (d - 1)))) continue;
        // speed along the normal: vmax s (parabolic, file) or -Re(K e^{iwt}) (Womersley)
        const double m = vmax * s[e] + vmax2 * s2[e];
        const double wx = io.n[0] * m * rho, wy = io.n[1] * m * rho, wz = io.n[2] * m * rho;
        const double correction =
            2. * Wt(d) * (wx * (double)CX[d] + wy * (double)CY[d] + wz * (double)CZ[d]) / CS2;
        stp(iolet_place(d, a.aout[d], slot, a.G, a.SI, r), 0, fpost[d] - correction);
      }
    }
  }
}

// Wall shear stress magnitude (Lattice.h:1122-1156 with the Pi tensor of
// :1353-1383) from the non-equilibrium change fpost - f.
__device__ __forceinline__ double wall_shear_stress(const StepArgs& a, uint32_t b, double tau, const double* f,
                                                    const double* fpost) {
  double g[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) g[j] = fpost[j] - f[j];
  const Sym3 s = second_moments(g);
  const double fac = -(tau - 0.5);
  const double p00 = s.xx * fac, p10 = s.yx * fac, p11 = s.yy * fac;
  const double p20 = s.zx * fac, p21 = s.zy * fac, p22 = s.zz * fac;
  const double n0 = (double)ldp(a.bnrm, b), n1 = (double)ldp(a.bnrm + a.SB, b),
               n2 = (double)ldp(a.bnrm + 2 * a.SB, b);
  double sv0 = p00 * n0;
  sv0 += p10 * n1;
  sv0 += p20 * n2;
  double sv1 = p10 * n0;
  sv1 += p11 * n1;
  sv1 += p21 * n2;
  double sv2 = p20 * n0;
  sv2 += p21 * n1;
  sv2 += p22 * n2;
  double sq = sv0 * sv0;
  sq += sv1 * sv1;
  sq += sv2 * sv2;
  double nn = sv0 * n0;
  nn += sv1 * n1;
  nn += sv2 * n2;
  return __builtin_sqrt(sq - nn * nn);
}

// Collision of one site from its moments: LBGK (LBGK.h:64-72), TRT
// (TRT.h:80-109) or LBGK with the relaxation time of LBGKLESSpongeLayer
// (Smagorinsky, :150-182, selected against the sponge's vTau of the site at
// slot by CalculateTau, :122-148); tau returns the site's.
template <int KERNEL>
__device__ __forceinline__ void collide_site(const StepArgs& a, const double* f, double rho, double mx, double my,
                                             double mz, uint32_t slot, double& tau, double* fpost) {
  const FeqPre pre = feq_pre(rho, mx, my, mz);
  double feq[Q];
  feq_all(pre, mx, my, mz, feq);
  double fneq[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) fneq[j] = f[j] - feq[j];
  tau = a.tau;
  if constexpr (KERNEL == HLB_KERNEL_LBGK) {
#pragma unroll
    for (int j = 0; j < Q; ++j) fpost[j] = f[j] + fneq[j] * a.omega;
  } else if constexpr (KERNEL == HLB_KERNEL_TRT) {
    // the (0,0) pair reduces to f0 + omega fneq0
    fpost[0] = f[0] + a.omega * fneq[0];
#pragma unroll
    for (int i = 1; i < Q; i += 2) {
      const int ib = i + 1;
      const double sym = a.half_omega * (fneq[i] + fneq[ib]);
      const double asym = a.half_omega_minus * (fneq[i] - fneq[ib]);
      fpost[i] = f[i] + sym + asym;
      fpost[ib] = f[ib] + sym - asym;
    }
  } else {
    const Sym3 s = second_moments(fneq);
    double q12 = s.xx * s.xx;
    q12 += s.yx * s.yx;
    q12 += s.zx * s.zx;
    q12 += s.yx * s.yx;
    q12 += s.yy * s.yy;
    q12 += s.zy * s.zy;
    q12 += s.zx * s.zx;
    q12 += s.zy * s.zy;
    q12 += s.zz * s.zz;
    q12 = __builtin_sqrt(q12);
    tau = 1. / 2. * (a.tau + __builtin_sqrt(a.tau * a.tau + a.les_k * q12));
    if (a.vtau != nullptr) {
      const double t = *a.sp_t;  // the step's time while the sponge lives, else -1
      if (t >= 0.0) {
        const double vt = ldp(a.vtau, slot);
        if (t <= a.sp_half) tau = vt == a.tau ? tau : vt;
        else tau = (tau - vt) * 2.0 / a.sp_life * t + (2.0 * vt - tau);
      }
    }
    const double om = -1.0 / tau;
#pragma unroll
    for (int j = 0; j < Q; ++j) fpost[j] = f[j] + fneq[j] * om;
  }
}

// The slab record of this lane's wavefront: four slabs per workgroup.
__device__ __forceinline__ uint32_t slab_record() {
  return xcd_tile() * (kBlock / kSlab) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
}

// B threads (B / 64 slabs) per workgroup; ORDER: the tile order
// (TileOrder).  NARROW: each pair of opposite planes fits 32-bit offsets from
// its lower plane (narrow_planes).
template <int KERNEL, bool FIRST, bool PROPS, int B = kBlock, int ORDER = kOrderXcd, int W = 0, bool NARROW = false,
          bool NT = false>
__global__ __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(W > 0 ? W : 1))) void step_fp64(StepArgs a) {
  if (wk_workgroup(a.wk, a.step)) return;
  Lane L;
  const uint32_t tile = tile_index<ORDER>(a.wk.groups);
  if (!slab_lane(a.bt, tile * (B / kSlab) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), L)) return;
  const uint32_t d = L.slot;
  Bnd bnd = no_bnd();
  if (L.boundary) bnd = load_bnd(a.bnd, L.b);
  double f[Q];
  if constexpr (FIRST) {
    // Initial condition or checkpoint: f is the pre-collision state itself.
#pragma unroll
    for (int j = 0; j < Q; ++j) f[j] = ldp(a.ain[j], d);
  } else {
    gather_site<NARROW>(a, L, f);
    if (L.boundary) boundary_fixup(a, d, L.b, bnd, f);
  }
  if (a.gz.pmask != nullptr) {
    // Sites the Guo-Zheng-Shi link kernel reads keep their pre-collision f.
    const uint64_t pm = uniform64(ldp(a.gz.pmask, L.r));
    if ((pm >> (threadIdx.x & 63u)) & 1u) {
      const uint32_t pi = (uint32_t)__builtin_amdgcn_readfirstlane(ldp(a.gz.pbase, L.r)) + lanes_below(pm);
#pragma unroll
      for (int j = 0; j < Q; ++j) stp(plane(a.P, a.gz.SP, j), pi, f[j]);
    }
  }

  // Moments and equilibrium (Lattice.h:933-948), collision.
  double rho, mx, my, mz;
  moments(f, rho, mx, my, mz);
  const double ux = mx / rho, uy = my / rho, uz = mz / rho;
  double tau;
  double fpost[Q];
  collide_site<KERNEL>(a, f, rho, mx, my, mz, d, tau, fpost);

  IoletIn io{};
  if (bnd.iolet != 0) io = load_iolet(a, bnd.gi);
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    if constexpr (NT) stp_nt(a.aout[j], d, fpost[j]);
    else stp(a.aout[j], d, fpost[j]);
  }

  if (bnd.iolet != 0) {
    const int bc = (int)bnd.gi < a.n_in ? a.inlet_bc : a.outlet_bc;
    iolet_links(a, d, bnd, io, bc, rho, ux, uy, uz, fpost);
    // InOutLetWK*::DoPreStreamCoupling: the coupling site's velocity.Dot(-normal).
    if (bnd.iolet & io.wk) {
      const double c = ux * -io.n[0] + uy * -io.n[1] + uz * -io.n[2];
      stp(a.wk_contrib, (uint32_t)ldp(a.wk_pos, bnd.ii), c);
    }
  }
  if constexpr (PROPS) {
    // BaseStreamer::UpdateMinsAndMaxes (BaseStreamer.h:88-120).
    stp(a.rho, d, rho);
    stp(a.u, d, ux);
    stp(plane(a.u, a.S, 1), d, uy);
    stp(plane(a.u, a.S, 2), d, uz);
    stp(a.wss, d, bnd.wall ? wall_shear_stress(a, L.b, tau, f, fpost) : DBL_MAX);
  }
}

// Materialises the pre-collision f (the reference's fOld entering the next
// step) into F, device order.
template <bool NARROW>
__global__ __launch_bounds__(kBlock) void gather_fp64(StepArgs a, double* __restrict__ F, int64_t S) {
  Lane L;
  if (!slab_lane(a.bt, slab_record(), L)) return;
  Bnd bnd = no_bnd();
  if (L.boundary) bnd = load_bnd(a.bnd, L.b);
  double f[Q];
  gather_site<NARROW>(a, L, f);
  if (L.boundary) boundary_fixup(a, L.slot, L.b, bnd, f);
#pragma unroll
  for (int j = 0; j < Q; ++j) stp(plane(F, S, j), L.slot, f[j]);
}

// The stress caches of MacroscopicPropertyCache (BaseStreamer.h:120-220)
// from the pre-collision state F (FP64, or FP32-shifted g with f = g + w):
// 17 planes of S doubles -- the full stress tensor (xx, xy, xz, yy, yz, zz;
// Lattice.h:1096-1111), von Mises stress (:983-1001), shear rate
// (:1159-1180), and at wall sites the traction (:1017-1027) with its
// tangential (:1045-1056) and normal (:1069-1079) projections (zero vectors
// elsewhere).  The collision and Pi tensor (:1353-1383) are the step's.
template <int KERNEL, typename T>
__global__ __launch_bounds__(kBlock) void stress_fp64(StepArgs a, const T* __restrict__ F, double* __restrict__ out) {
  Lane L;
  if (!slab_lane(a.bt, slab_record(), L)) return;
  const uint32_t d = L.slot;
  double f[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    if constexpr (sizeof(T) == 8) f[j] = (double)ldp(plane(F, a.S, j), d);
    else f[j] = (double)ldp(plane(F, a.S, j), d) + Wt(j);
  }
  double rho, mx, my, mz;
  moments(f, rho, mx, my, mz);
  double tau;
  double fpost[Q];
  collide_site<KERNEL>(a, f, rho, mx, my, mz, d, tau, fpost);
  double g[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) g[j] = fpost[j] - f[j];
  const Sym3 s = second_moments(g);
  const double fac = -(tau - 0.5);
  const double p00 = s.xx * fac, p10 = s.yx * fac, p11 = s.yy * fac;
  const double p20 = s.zx * fac, p21 = s.zy * fac, p22 = s.zz * fac;
  const double pi[3][3] = {{p00, p10, p20}, {p10, p11, p21}, {p20, p21, p22}};
  // stress tensor: -Pi, minus the pressure (rho - 1) Cs2 on the diagonal
  double sig[3][3];
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) sig[r][c] = -1.0 * pi[r][c];
  const double pressure = (rho - 1) * CS2;
#pragma unroll
  for (int r = 0; r < 3; ++r) sig[r][r] += -pressure;
  const double ten[6] = {sig[0][0], sig[0][1], sig[0][2], sig[1][1], sig[1][2], sig[2][2]};
#pragma unroll
  for (int k = 0; k < 6; ++k) stp(plane(out, a.S, k), d, ten[k]);
  // von Mises stress
  const double dxy = p00 - p11, dyz = p11 - p22, dzx = p22 - p00;
  const double t1 = dxy * dxy + dyz * dyz + dzx * dzx;
  const double t2 = pi[0][1] * pi[0][1] + pi[1][2] * pi[1][2] + pi[2][0] * pi[2][0];
  stp(plane(out, a.S, 6), d, __builtin_sqrt(0.5 * (t1 + 6.0 * t2)));
  // shear rate
  double sr = 0.0;
#pragma unroll
  for (int r = 0; r < 3; ++r)
#pragma unroll
    for (int c = 0; c < 3; ++c) sr += pi[r][c] * pi[r][c];
  sr = __builtin_sqrt(sr) / (-2.0 * CS2 * rho);
  sr /= (tau - 0.5);
  stp(plane(out, a.S, 7), d, sr);
  // traction and its projections at wall sites
  double tr[3] = {0.0, 0.0, 0.0}, tt[3] = {0.0, 0.0, 0.0}, tn[3] = {0.0, 0.0, 0.0};
  if (L.boundary && load_bnd(a.bnd, L.b).wall) {
    const double n[3] = {(double)ldp(a.bnrm, L.b), (double)ldp(a.bnrm + a.SB, L.b),
                         (double)ldp(a.bnrm + 2 * a.SB, L.b)};
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      tr[r] = 0.0;
#pragma unroll
      for (int c = 0; c < 3; ++c) tr[r] += sig[r][c] * n[c];
    }
    const double mag = tr[0] * n[0] + tr[1] * n[1] + tr[2] * n[2];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      tt[r] = tr[r] - n[r] * mag;
      tn[r] = n[r] * mag;
    }
  }
#pragma unroll
  for (int r = 0; r < 3; ++r) {
    stp(plane(out, a.S, 8 + r), d, tr[r]);
    stp(plane(out, a.S, 11 + r), d, tt[r]);
    stp(plane(out, a.S, 14 + r), d, tn[r]);
  }
}

// GuoZhengShiDelegate::StreamLink (GuoZhengShiDelegate.h:123-294), one
// thread per GZS wall link, from the pre-collision f the step stored in P:
// the wall node's momentum is this site's scaled by 1 - 1/q, interpolated
// (q < 0.75) with the next fluid site out or a velocity iolet's profile; its
// f_neq likewise (next site only); the node is collided with the run's
// kernel and its value in direction i = INV[d] is the site's next input.
template <int KERNEL>
__global__ __launch_bounds__(kBlock) void gzs_links_fp64(StepArgs a, const GzsLink* __restrict__ links, int n,
                                                         const double* __restrict__ vmax, double* __restrict__ GW) {
  const int e = blockIdx.x * kBlock + threadIdx.x;
  if (e >= n) return;
  const GzsLink lk = links[e];
  const int d = lk.dir, i = INV[d];
  const double q = (double)lk.q;
  double f[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) f[j] = ldp(plane(a.P, a.gz.SP, j), (uint32_t)lk.site_p);
  double rho, mx, my, mz;
  moments(f, rho, mx, my, mz);
  double feq[Q], fneq[Q];
  feq_all(feq_pre(rho, mx, my, mz), mx, my, mz, feq);
#pragma unroll
  for (int j = 0; j < Q; ++j) fneq[j] = f[j] - feq[j];
  const double fac = 1. - 1. / q;
  double wm[3] = {mx * fac, my * fac, mz * fac};
  if (lk.mode == 2) {
    double g[Q];
#pragma unroll
    for (int j = 0; j < Q; ++j) g[j] = ldp(plane(a.P, a.gz.SP, j), (uint32_t)lk.nb_p);
    double nr, nx, ny, nz;
    moments(g, nr, nx, ny, nz);
    const double nv[3] = {nx / nr, ny / nr, nz / nr};
    double gfeq[Q];
    feq_all(feq_pre(nr, nx, ny, nz), nx, ny, nz, gfeq);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double second = nv[c] * (q - 1) / (q + 1);
      wm[c] = q * wm[c] + (1. - q) * rho * second;
    }
#pragma unroll
    for (int j = 0; j < Q; ++j) fneq[j] = q * fneq[j] + (1. - q) * (g[j] - gfeq[j]);
  } else if (lk.mode == 3) {
    const double sp = ldp(vmax, (uint32_t)lk.gi) * lk.s + ldp(a.io_vmax2, (uint32_t)lk.gi) * lk.s2;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double v = ldp(a.io_n, 3u * lk.gi + c) * sp;
      const double second = v * (q - 1) / (q + 1);
      wm[c] = q * wm[c] + (1. - q) * rho * second;
    }
  }
  double weq[Q];
  feq_all(feq_pre(rho, wm[0], wm[1], wm[2]), wm[0], wm[1], wm[2], weq);
  double fw[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) fw[j] = weq[j] + fneq[j];
  double val;
  if constexpr (KERNEL == HLB_KERNEL_TRT) {
    const int lo = i < INV[i] ? i : INV[i], hi = i < INV[i] ? INV[i] : i;
    const double sym = a.half_omega * (fneq[lo] + fneq[hi]);
    const double asym = a.half_omega_minus * (fneq[lo] - fneq[hi]);
    val = i == lo ? fw[lo] + sym + asym : fw[hi] + sym - asym;
  } else {
    val = fw[i] + fneq[i] * a.omega;
  }
  stp(GW, (uint32_t)e, val);
}

// The slot each lane gathers direction J from (the lane's own slot for a
// wall or iolet link), 18 planes of S: the step kernels' addressing, exported
// so the host can compare it with the reference's neighbour table.
template <int J = 1>
__device__ __forceinline__ void upstream_all(const Lane& L, uint32_t* out, int64_t S) {
  if constexpr (J < Q) {
    stp(plane(out, S, J - 1), L.slot, upstream_slot<J>(L));
    upstream_all<J + 1>(L, out, S);
  }
}

__global__ __launch_bounds__(kBlock) void upstream_table(BrickTables bt, uint32_t* __restrict__ out, int64_t S) {
  Lane L;
  if (!slab_lane(bt, slab_record(), L)) return;
  upstream_all(L, out, S);
}

// Monitors over the fluid sites' property fields (the last step that filled
// them): min rho, max rho, max |u| -- the IncompressibilityChecker's
// DensityTracker (IncompressibilityChecker.hpp:170-195, |u| as
// Vector3D::GetMagnitude) -- and the total mass sum rho.  Pass 1 reduces each
// workgroup in a fixed tree order into partial[wg]; pass 2 reduces the
// partials in order, so the sum is reproducible run to run.
struct Mon {
  double lo, hi, umax, mass;
};

__device__ __forceinline__ Mon mon_join(Mon a, Mon b) {
  return Mon{__builtin_fmin(a.lo, b.lo), __builtin_fmax(a.hi, b.hi), __builtin_fmax(a.umax, b.umax), a.mass + b.mass};
}

__device__ __forceinline__ Mon mon_wave(Mon m) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    Mon o{__shfl_xor(m.lo, off, 64), __shfl_xor(m.hi, off, 64), __shfl_xor(m.umax, off, 64),
          __shfl_xor(m.mass, off, 64)};
    m = mon_join(m, o);
  }
  return m;
}

__global__ __launch_bounds__(kBlock) void monitor_pass1(BrickTables bt, const double* __restrict__ rho,
                                                        const double* __restrict__ u, int64_t S,
                                                        Mon* __restrict__ partial) {
  __shared__ Mon w[kBlock / 64];
  Mon m{DBL_MAX, -DBL_MAX, 0.0, 0.0};
  Lane L;
  if (slab_lane(bt, slab_record(), L)) {
    const double r = ldp(rho, L.slot);
    const double x = ldp(u, L.slot), y = ldp(plane(u, S, 1), L.slot), z = ldp(plane(u, S, 2), L.slot);
    m = Mon{r, r, __builtin_sqrt(x * x + y * y + z * z), r};
  }
  m = mon_wave(m);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    Mon t = w[0];
    for (int i = 1; i < kBlock / 64; ++i) t = mon_join(t, w[i]);
    partial[blockIdx.x] = t;
  }
}

__global__ __launch_bounds__(kBlock) void monitor_pass2(const Mon* __restrict__ partial, int n, double* __restrict__ out,
                                                        bool signal) {
  __shared__ Mon w[kBlock / 64];
  Mon m{DBL_MAX, -DBL_MAX, 0.0, 0.0};
  // each lane folds a contiguous run, in order
  const int per = (n + kBlock - 1) / kBlock;
  for (int i = threadIdx.x * per; i < n && i < (int)(threadIdx.x + 1) * per; ++i) m = mon_join(m, partial[i]);
  m = mon_wave(m);
  if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    Mon t = w[0];
    for (int i = 1; i < kBlock / 64; ++i) t = mon_join(t, w[i]);
    out[0] = t.lo;
    out[1] = t.hi;
    out[2] = t.umax;
    out[3] = t.mass;
    // a host that sees out[4] set has the four before it (0.5 us, which a caller
    // that waits for the stream need not spend)
    if (signal) __hip_atomic_store(out + 4, 1.0, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__global__ __launch_bounds__(kBlock) void fill_planes_fp64(double* __restrict__ F, int64_t N, int64_t S,
                                                           const double* __restrict__ vals) {
  const int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (k >= N) return;
#pragma unroll
  for (int j = 0; j < Q; ++j) F[(int64_t)j * S + k] = vals[j];
}

// StabilityTester: flag any !(f > 0) among the fluid sites' distributions.
__global__ __launch_bounds__(kBlock) void unstable_fp64(BrickTables bt, const double* __restrict__ F, int64_t S,
                                                        int* __restrict__ flag) {
  Lane L;
  if (!slab_lane(bt, slab_record(), L)) return;
  bool bad = false;
#pragma unroll
  for (int j = 0; j < Q; ++j) bad |= !(ldp(plane(F, S, j), L.slot) > 0.0);
  if (bad) *flag = 1;
}

// First row of a sequence: the ghost densities its first step reads
// (InOutLetWK*::DoComms, density <- densityNew).  One thread per iolet.
__global__ __launch_bounds__(256) void wk_start(const WkRef* __restrict__ refs, int n) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const WkRef ref = refs[r];
  ref.io_dens[ref.g] = ref.w->densityNew;
}

// End of a sequence: the sum of its last step's flux terms, which the next
// step's DoComms scales.  One wavefront per iolet.
__global__ __launch_bounds__(64) void wk_flush(const WkRef* __restrict__ refs, int last) {
  const WkRef ref = refs[blockIdx.x];
  const double sum = wk_flux_sum(ref, last);
  if (threadIdx.x != 0) return;
  ref.w->flowRateNew = sum;
  ref.w->siteCount = (double)(ref.w->list_end - ref.w->list_begin);
}

}  // namespace

hipError_t launch_wk_start(const WkRef* refs, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(wk_start, dim3((n + 255) / 256), dim3(256), 0, s, refs, n);
  return hipGetLastError();
}

hipError_t launch_wk_flush(const WkRef* refs, int n, int last, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(wk_flush, dim3(n), dim3(64), 0, s, refs, last);
  return hipGetLastError();
}

unsigned grid_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

// Site grids are padded to a multiple of the XCD count for the remapping.
// Workgroups of four slabs, padded to a multiple of the XCD count.
static unsigned slab_grid(int64_t nslab) {
  const int64_t wg = (nslab + kBlock / kSlab - 1) / (kBlock / kSlab);
  return (unsigned)((wg + kXcds - 1) / kXcds * kXcds);
}

// 32-bit element offsets from the lower plane of each opposite pair cover
// both planes (the byte offset i * 8 stays below 2^32), and the planes are one
// allocation.  Lattices above 2^28 slots, and every lattice when the handle
// asks for it (a test switch), pick the plane with the 64-bit address.
static bool narrow_planes(const StepArgs& a) {
  return !a.general_gather && 2 * a.S <= (int64_t(1) << 29) && a.ain[18] == a.ain[0] + 18 * a.S;
}

// Steady-state steps in launch shape `variant` (as the FP32 kernel's).
template <int KN, bool NARROW>
void launch_variant_fp64(const StepArgs& a, int variant, hipStream_t s) {
  const LaunchShape l = launch_shape(variant, false);
  const int per = shape_slabs(l);
  const dim3 grid(a.wk.groups + shape_grid(l, (a.bt.nslab + per - 1) / per));
  const unsigned lds = shape_lds(l);
#define HLB_V(B, O, W)                                                                                   \
  if (l.nt)                                                                                              \
    hipLaunchKernelGGL((step_fp64<KN, false, false, B, O, W, NARROW, true>), grid, dim3(B), lds, s, a);  \
  else                                                                                                   \
    hipLaunchKernelGGL((step_fp64<KN, false, false, B, O, W, NARROW, false>), grid, dim3(B), lds, s, a)
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
  // the FP64 kernel fits 4 waves per SIMD as compiled; levels 4, 5 ask for 5, 6
  switch (l.level) {
    case 4: HLB_SHAPES(5); break;
    case 5: HLB_SHAPES(6); break;
    default: HLB_SHAPES(0); break;
  }
#undef HLB_SHAPES
#undef HLB_ORDERS
#undef HLB_V
}

hipError_t launch_step_fp64(const StepArgs& a, int kernel, bool first, bool props, int variant, hipStream_t s) {
  if (a.bt.nslab <= 0) return hipSuccess;
  const bool narrow = narrow_planes(a);
  if (!first && !props) {
#define HLB_K(KN)                                          \
  if (narrow) launch_variant_fp64<KN, true>(a, variant, s); \
  else launch_variant_fp64<KN, false>(a, variant, s);
    switch (kernel) {
      case HLB_KERNEL_LBGK: HLB_K(HLB_KERNEL_LBGK); break;
      case HLB_KERNEL_TRT: HLB_K(HLB_KERNEL_TRT); break;
      default: HLB_K(HLB_KERNEL_LES); break;
    }
#undef HLB_K
    return hipGetLastError();
  }
  // one-slab tiles in XCD order, the store policy of the variant
  const LaunchShape l{kSlab, kOrderXcd, 0, 1, launch_shape(variant, false).nt};
  const dim3 grid(a.wk.groups + shape_grid(l, a.bt.nslab)), block(kSlab);
#define HLB_LAUNCH(KN, FI, PR, NA)                                                                       \
  do {                                                                                                   \
    if (l.nt) hipLaunchKernelGGL((step_fp64<KN, FI, PR, kSlab, kOrderXcd, 0, NA, true>), grid, block, 0, s, a); \
    else hipLaunchKernelGGL((step_fp64<KN, FI, PR, kSlab, kOrderXcd, 0, NA, false>), grid, block, 0, s, a);     \
  } while (0)
#define HLB_KSEL(KN)                                   \
  if (first) {                                         \
    if (props) HLB_LAUNCH(KN, true, true, false);      \
    else HLB_LAUNCH(KN, true, false, false);           \
  } else {                                             \
    if (narrow) HLB_LAUNCH(KN, false, true, true);     \
    else HLB_LAUNCH(KN, false, true, false);           \
  }
  switch (kernel) {
    case HLB_KERNEL_LBGK: HLB_KSEL(HLB_KERNEL_LBGK); break;
    case HLB_KERNEL_TRT: HLB_KSEL(HLB_KERNEL_TRT); break;
    default: HLB_KSEL(HLB_KERNEL_LES); break;
  }
#undef HLB_KSEL
#undef HLB_LAUNCH
  return hipGetLastError();
}

hipError_t launch_gzs_fp64(const StepArgs& a, int kernel, const GzsLink* links, int n, const double* vmax,
                           double* GW, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const dim3 grid((n + kBlock - 1) / kBlock), block(kBlock);
  if (kernel == HLB_KERNEL_TRT) hipLaunchKernelGGL(gzs_links_fp64<HLB_KERNEL_TRT>, grid, block, 0, s, a, links, n, vmax, GW);
  else hipLaunchKernelGGL(gzs_links_fp64<HLB_KERNEL_LBGK>, grid, block, 0, s, a, links, n, vmax, GW);
  return hipGetLastError();
}

hipError_t launch_upstream_table(const BrickTables& bt, uint32_t* out, int64_t S, hipStream_t s) {
  if (bt.nslab <= 0) return hipSuccess;
  hipLaunchKernelGGL(upstream_table, dim3(slab_grid(bt.nslab)), dim3(kBlock), 0, s, bt, out, S);
  return hipGetLastError();
}

size_t monitor_scratch(int64_t nslab) { return sizeof(Mon) * std::max<size_t>(1, slab_grid(nslab)); }

hipError_t launch_monitor(const BrickTables& bt, const double* rho, const double* u, int64_t S, void* scratch,
                          double* out, bool signal, hipStream_t s) {
  if (bt.nslab <= 0) return hipSuccess;
  const unsigned grid = slab_grid(bt.nslab);
  Mon* part = static_cast<Mon*>(scratch);
  hipLaunchKernelGGL(monitor_pass1, dim3(grid), dim3(kBlock), 0, s, bt, rho, u, S, part);
  hipLaunchKernelGGL(monitor_pass2, dim3(1), dim3(kBlock), 0, s, part, (int)grid, out, signal);
  return hipGetLastError();
}

hipError_t launch_stress_fp64(const StepArgs& a, int kernel, const void* F, bool fp32, double* out, hipStream_t s) {
  if (a.bt.nslab <= 0) return hipSuccess;
  const dim3 grid(slab_grid(a.bt.nslab)), block(kBlock);
#define HLB_S(KN)                                                                                          \
  if (fp32) hipLaunchKernelGGL((stress_fp64<KN, float>), grid, block, 0, s, a, static_cast<const float*>(F), out); \
  else hipLaunchKernelGGL((stress_fp64<KN, double>), grid, block, 0, s, a, static_cast<const double*>(F), out)
  switch (kernel) {
    case HLB_KERNEL_LBGK: HLB_S(HLB_KERNEL_LBGK); break;
    case HLB_KERNEL_TRT: HLB_S(HLB_KERNEL_TRT); break;
    default: HLB_S(HLB_KERNEL_LES); break;
  }
#undef HLB_S
  return hipGetLastError();
}

hipError_t launch_gather_fp64(const StepArgs& a, double* F, int64_t S, hipStream_t s) {
  if (a.bt.nslab <= 0) return hipSuccess;
  const dim3 grid(slab_grid(a.bt.nslab)), block(kBlock);
  if (narrow_planes(a)) hipLaunchKernelGGL(gather_fp64<true>, grid, block, 0, s, a, F, S);
  else hipLaunchKernelGGL(gather_fp64<false>, grid, block, 0, s, a, F, S);
  return hipGetLastError();
}

hipError_t launch_fill_fp64(double* F, int64_t N, int64_t S, const double* vals, hipStream_t s) {
  if (N <= 0) return hipSuccess;
  hipLaunchKernelGGL(fill_planes_fp64, dim3(grid_for(N)), dim3(kBlock), 0, s, F, N, S, vals);
  return hipGetLastError();
}

hipError_t launch_unstable_fp64(const BrickTables& bt, const double* F, int64_t S, int* flag, hipStream_t s) {
  if (bt.nslab <= 0) return hipSuccess;
  hipLaunchKernelGGL(unstable_fp64, dim3(slab_grid(bt.nslab)), dim3(kBlock), 0, s, bt, F, S, flag);
  return hipGetLastError();
}

}  // namespace hlb
