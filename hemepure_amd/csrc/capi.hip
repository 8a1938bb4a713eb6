// capi.hip -- the extern "C" boundary: handle lifecycle, device buffers,
// iolet bookkeeping and the step driver.
//
// A handle plays the roles of the reference's LatticeData (tables and f
// arrays), LBM (kernel/streamer selection and the phase sequence) and the two
// BoundaryValues objects (iolet state), for one GPU.  Every array crossing the
// boundary is in the reference's class-major site order; the device works in
// natural block order (see lbm_kernels.h) and the handle maps between them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <atomic>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "../../include/hemepure_amd.h"
#include "d3q19.h"
#include "errors.h"
#include "handle.h"
#include "iolet_math.h"
#include "lattice.h"
#include "lbm_kernels.h"
#include "transfer.h"

namespace hlb {

std::string& last_error() {
  thread_local std::string msg;
  return msg;
}

}  // namespace hlb

namespace hlb {
namespace {

// The lattice direction closest to the iolet normal: the same std::sort over
// |c_k/|c_k| - n|^2 as NashZerothOrderPressureDelegate.h:95-116.
int direction_closest_to(const double n[3]) {
  std::array<int, Q> dirs;
  std::array<double, Q> dist;
  for (int k = 0; k < Q; ++k) {
    double cx = CX[k], cy = CY[k], cz = CZ[k];
    if (!(cx == 0.0 && cy == 0.0 && cz == 0.0)) {
      const double mag = std::sqrt(cx * cx + cy * cy + cz * cz);
      cx /= mag;
      cy /= mag;
      cz /= mag;
    }
    const double ex = cx - n[0], ey = cy - n[1], ez = cz - n[2];
    dist[k] = ex * ex + ey * ey + ez * ez;
    dirs[k] = k;
  }
  std::sort(dirs.begin(), dirs.end(), [&dist](int i, int j) { return dist[i] < dist[j]; });
  return dirs[0];
}

// InOutLetCosine::GetDensity (src/lb/iolets/InOutLetCosine.cc:37-54) at the
// 0-indexed step t0.
double cosine_density(const HostIolet& io, uint64_t t0) {
  const double w = 2.0 * kPi / io.d.period;
  const double target = io.d.density_mean + io.d.density_amp * std::cos(w * t0 + io.d.phase);
  const uint32_t warm = (uint32_t)io.d.warmup;
  if (t0 >= warm) return target;
  const double f = ((double)t0) / ((double)warm);
  return f * target + (1. - f) * io.minSimDensity;
}

// Points the arguments at the per-step values of step s of a sequence whose
// rows are at `rows`.
void step_rows(const hlb_lattice* h, StepArgs& a, const double* rows, int64_t s) {
  const int64_t nio = h->iolet_count();
  a.io_dens = rows + s * h->row();
  a.io_vmax = a.io_dens + nio;
  a.io_vmax2 = a.io_dens + 2 * nio;
  a.sp_t = a.io_dens + 3 * nio;
}

StepArgs make_args(hlb_lattice* h, const double* ain, double* aout) {
  StepArgs a{};
  for (int j = 0; j < Q; ++j) {
    a.ain[j] = ain ? ain + (size_t)j * h->S : nullptr;
    a.aout[j] = aout ? aout + (size_t)j * h->S : nullptr;
  }
  a.bt = h->tables();
  a.gz = h->gz_tables();
  a.P = h->P64.p;
  a.GW = h->GW64.p;
  a.bnd = h->bnd.p;
  a.bq = h->bq.p;
  a.bnrm = h->bnrm.p;
  a.G = h->G.p;
  a.ladd_s = h->ladd_s.p;
  a.ladd_s2 = h->ladd_s.p ? h->ladd_s.p + (size_t)18 * h->SI : nullptr;
  a.rho = h->rho.p;
  a.u = h->u.p;
  a.wss = h->wss.p;
  a.io_n = h->io_n.p;
  a.wk_bit = h->wk_bit.p;
  a.wk_pos = h->wk_pos.p;
  a.wk_contrib = h->wk_contrib.p;
  a.N = h->L.N;
  a.S = h->S;
  a.SB = h->SB;
  a.SI = h->SI;
  a.n_in = h->n_in;
  a.inlet_bc = h->params.inlet_bc;
  a.outlet_bc = h->params.outlet_bc;
  a.tau = h->params.tau;
  a.omega = h->omega;
  a.half_omega = h->half_omega;
  a.half_omega_minus = h->half_omega_minus;
  a.les_k = h->les_k;
  a.general_gather = h->general_gather ? 1 : 0;
  a.vtau = h->sponge_life > 0 ? h->vtau64.p : nullptr;
  step_rows(h, a, h->rows(), 0);
  a.sp_half = (double)(h->sponge_life / 2);
  a.sp_life = (double)h->sponge_life;
  return a;
}

// The profile factors (s, s2) of a velocity iolet at x: speed = vmax s +
// vmax2 s2 along the normal.  Parabolic and file profiles: 1 - r^2/a^2
// (InOutLetParabolicVelocity.cc:30-52, InOutLetFileVelocity.cc:93-109),
// HLB_ERANGE outside the radius as the reference's exit(16); Womersley:
// -Re K and Im K, so that vmax s + vmax2 s2 = -Re(K e^{iwt}).
int velocity_factors(const HostIolet& io, const double x[3], double& s, double& s2) {
  if (io.d.kind == HLB_IOLET_WOMERSLEY) {
    double kre, kim;
    womersley_coefficient(io.d.position, io.n, io.d.radius, io.d.period, io.d.womersley_number,
                          io.d.pressure_gradient_amplitude, x, &kre, &kim);
    s = -kre;
    s2 = kim;
    return HLB_OK;
  }
  const double dx = x[0] - io.d.position[0], dy = x[1] - io.d.position[1], dz = x[2] - io.d.position[2];
  const double z = dx * io.n[0] + dy * io.n[1] + dz * io.n[2];
  const double rSq = (dx * dx + dy * dy + dz * dz) - z * z;
  const double r2a2 = rSq / (io.d.radius * io.d.radius);
  if (r2a2 > 1.0) {
    char buf[200];
    std::snprintf(buf, sizeof buf, "An IOLET site with r = %lf lies outside the IOLET radius %lf.", std::sqrt(rSq),
                  io.d.radius);
    return fail(HLB_ERANGE, buf);
  }
  s = 1. - r2a2;
  s2 = 0.0;
  return HLB_OK;
}

// Ghost density (Nash) and the speed factors (Ladd, GZS) of every iolet at
// 1-indexed step t: a velocity iolet's speed along its normal at a link is
// vmax * s + vmax2 * s2 with the link's profile factors s, s2.
int iolet_values(const hlb_lattice* h, int64_t t, double* dens, double* vmax, double* vmax2) {
  const int nio = (int)h->iolets.size();
  for (int g = 0; g < nio; ++g) {
    const HostIolet& io = h->iolets[g];
    dens[g] = 1.0;
    vmax[g] = 0.0;
    vmax2[g] = 0.0;
    switch (io.d.kind) {
      case HLB_IOLET_COSINE: dens[g] = cosine_density(io, (uint64_t)(t - 1)); break;
      case HLB_IOLET_FILEPRES:
        // InOutLetFile::GetDensity(Get0IndexedTimeStep()) (InOutLetFile.h:56-59)
        if (t - 1 >= (int64_t)io.table.size())
          return fail(HLB_ERANGE, "pressure table of iolet " + std::to_string(g) + " ends before step " +
                                      std::to_string(t));
        dens[g] = io.table[t - 1];
        break;
      case HLB_IOLET_PARABOLIC: {
        // InOutLetParabolicVelocity.cc:47-52
        double max = io.d.max_speed;
        const uint32_t warm = (uint32_t)io.d.warmup;
        if ((uint64_t)t < warm) max *= (uint64_t)t / double(warm);
        vmax[g] = max;
        break;
      }
      case HLB_IOLET_FILEVEL:
        if (t >= (int64_t)io.table.size())
          return fail(HLB_ERANGE, "velocity table of iolet " + std::to_string(g) + " ends before step " +
                                      std::to_string(t));
        vmax[g] = io.table[t];
        break;
      case HLB_IOLET_WOMERSLEY: {
        // the time factor exp(i omega t) of InOutLetWomersleyVelocity.cc:35-37
        womersley_time_factor(io.d.period, t, &vmax[g], &vmax2[g]);
        break;
      }
      default: break;
    }
  }
  return HLB_OK;
}

int side_iolet(const hlb_lattice* h, int64_t k) {
  const int c = h->L.collision_class(k);
  return (c == 2 || c == 4) ? h->L.ioletId[k] : h->n_in + h->L.ioletId[k];
}

// The slab layout: the site grid cut into 8^3 tiles (independent of the
// geometry's own block size), occupied tiles numbered in tile order (z
// fastest) as bricks, each brick's x layers with a fluid site as slabs,
// enumerated brick by brick (TILE) or layer by layer (LAYER).  A slab's fluid
// lanes (lane = y * 8 + z) take consecutive slots from its base; bases are
// rounded up to kSlabAlign.  Boundary and iolet sites are numbered in slot
// order.  Each slab's record lists the masks and bases of the slabs its lanes
// pull from.
//
// Why LAYER: the face lanes of a slab's rows (y = 0 or 7, 32 B of a 128 B
// line in FP32) are read by the slab of the y-neighbouring brick, the rest by
// the slab downstream in its own brick.  Under the XCD-contiguous launch
// order an XCD walks its slabs in storage order, and the line is fetched once
// only if both readers come within the XCD's 4 MiB L2 window: about 431
// slabs at 2 x 19 x 256 B of FP32 rows read and written per slab.  In TILE
// order the y neighbour is one occupied z-row of bricks, times their layers,
// later; LAYER order divides that by the layer count (the x neighbours it
// moves apart read whole rows, which no other slab shares).  Measured on
// MI355X: the 65M-site vessel tree (median y distance 628 slabs) reads 92
// instead of 102 B per FP32 site update and steps 5% faster; lattices below
// the window (the Y-bifurcation, 229 to 463 slabs) keep TILE, which is as
// fast or faster there.
constexpr int64_t kL2WindowSlabs = 431;

// Why sections: in XCD order each XCD takes one eighth of the slabs.  In tile
// order (x slowest) the eighths of a vessel that runs along z or y are slices
// along it: those at its sides are mostly boundary slabs, which take about
// twice as long, and the XCDs in the middle wait.  AUTO therefore enumerates
// such a vessel in sections of kSectionBricks bricks along its longest axis,
// tile order within, where XCD order is what a lattice is launched in and its
// steps are long enough for it to show: distributions between a quarter of the
// Infinity Cache and all of it.  Measured on MI355X, tile order / sections: the
// 0.70M-site Y-bifurcation (z) FP64 44.9 / 41.6-42.1 us, FP32 27.0 / 25.8-26.1;
// beyond the cache nothing or a loss (3.0M-site tree 206.6 / 206.5, 1.9M-site
// pipe 119.0 / 119.2, 20-pipe ensemble 67.7 / 69.7).
constexpr int64_t kSectionBricks = 8;
bool sections_pay(int64_t sites, bool fp32) {
  const int64_t bytes = distribution_bytes(sites, fp32);
  return bytes > kInfinityCacheBytes / 4 && bytes <= kInfinityCacheBytes;
}

// m's positions moved by BY, for those that stay within the slab.
template <int BY>
uint64_t moved(uint64_t m) {
  if constexpr (BY >= 64 || BY <= -64) return 0;
  else if constexpr (BY >= 0) return m >> BY;
  else return m << -BY;
}

// Fluid upstream positions of a slab's sites in directions J and up, from the
// masks of the reachable slabs (upstream_pos on the host).
template <int J = 1>
int fluid_neighbours(const SlabRec& R) {
  if constexpr (J == Q) {
    return 0;
  } else {
    constexpr int ox = -CX[J], oy = -CY[J], oz = -CZ[J], by = 8 * oy + oz;
    constexpr uint64_t Y = oy == 0 ? 0 : oy > 0 ? 0xffull << 56 : 0xffull;
    constexpr uint64_t Z = oz == 0 ? 0 : oz > 0 ? 0x8080808080808080ull : 0x0101010101010101ull;
    uint64_t f = moved<by>(R.fm[reach_entry(ox, 0, 0)]) & ~(Y | Z);
    if constexpr (oy != 0) f |= moved<by - 64 * oy>(R.fm[reach_entry(ox, oy, 0)]) & Y & ~Z;
    if constexpr (oz != 0) f |= moved<by - 8 * oz>(R.fm[reach_entry(ox, 0, oz)]) & Z & ~Y;
    if constexpr (oy != 0 && oz != 0) f |= moved<by - 64 * oy - 8 * oz>(R.fm[reach_entry(ox, oy, oz)]) & Y & Z;
    return __builtin_popcountll(f & R.fm[reach_entry(0, 0, 0)]) + fluid_neighbours<J + 1>(R);
  }
}

void device_order(hlb_lattice* h, int order) {
  const HostLattice& L = h->L;
  const int64_t N = L.N;
  const int64_t ntx = ((int64_t)L.blocks[0] * L.bs + 7) / 8, nty = ((int64_t)L.blocks[1] * L.bs + 7) / 8,
                ntz = ((int64_t)L.blocks[2] * L.bs + 7) / 8;
  auto tile_of = [&](int64_t x, int64_t y, int64_t z) { return (x * nty + y) * ntz + z; };
  std::vector<int32_t> brickOf((size_t)(ntx * nty * ntz), -1);
  parallel_ranges(N, [&](int, int64_t lo, int64_t hi) {
    for (int64_t k = lo; k < hi; ++k) {
      int32_t* b = &brickOf[(size_t)tile_of(L.coords[3 * k] >> 3, L.coords[3 * k + 1] >> 3, L.coords[3 * k + 2] >> 3)];
      if (__atomic_load_n(b, __ATOMIC_RELAXED) != 0) __atomic_store_n(b, 0, __ATOMIC_RELAXED);
    }
  });
  std::vector<int64_t> brickTile;
  for (size_t t = 0; t < brickOf.size(); ++t)
    if (brickOf[t] >= 0) brickTile.push_back((int64_t)t);
  if (order == HLB_ORDER_AUTO && sections_pay(N, h->params.precision == HLB_FP32_SHIFTED)) {
    int64_t lo[3] = {ntx, nty, ntz}, hi[3] = {-1, -1, -1};
    auto axis_of = [&](int64_t t, int a) { return a == 0 ? t / (nty * ntz) : a == 1 ? (t / ntz) % nty : t % ntz; };
    for (const int64_t t : brickTile)
      for (int a = 0; a < 3; ++a) {
        lo[a] = std::min(lo[a], axis_of(t, a));
        hi[a] = std::max(hi[a], axis_of(t, a));
      }
    int along = 0;
    for (int a = 1; a < 3; ++a)
      if (hi[a] - lo[a] > hi[along] - lo[along]) along = a;
    if (along != 0)
      std::stable_sort(brickTile.begin(), brickTile.end(), [&](int64_t s, int64_t t) {
        return axis_of(s, along) / kSectionBricks < axis_of(t, along) / kSectionBricks;
      });
  }
  for (size_t i = 0; i < brickTile.size(); ++i) brickOf[(size_t)brickTile[i]] = (int32_t)i;
  const int64_t NBr = (int64_t)brickTile.size();
  h->nbrick = NBr;
  constexpr int64_t kBrickGrain = kGrain / kBrickSites;
  // the site at each position of each brick
  RawVector<int32_t> at;
  at.resize((size_t)NBr * kBrickSites);
  parallel_ranges(NBr, [&](int, int64_t lo, int64_t hi) {
    std::fill(at.begin() + lo * kBrickSites, at.begin() + hi * kBrickSites, -1);
  }, kBrickGrain);
  parallel_ranges(N, [&](int, int64_t lo, int64_t hi) {
    for (int64_t k = lo; k < hi; ++k) {
      const int32_t x = L.coords[3 * k], y = L.coords[3 * k + 1], z = L.coords[3 * k + 2];
      const int64_t brick = brickOf[(size_t)tile_of(x >> 3, y >> 3, z >> 3)];
      at[(size_t)brick * kBrickSites + ((x & 7) * 8 + (y & 7)) * 8 + (z & 7)] = (int32_t)k;
    }
  });
  // fluid masks of every layer of every brick
  std::vector<uint64_t> fmAll((size_t)NBr * 8, 0);
  parallel_ranges(NBr * 8, [&](int, int64_t lo, int64_t hi) {
    for (int64_t i = lo; i < hi; ++i)
      for (int lane = 0; lane < kSlab; ++lane)
        if (at[(size_t)i * kSlab + lane] >= 0) fmAll[(size_t)i] |= 1ull << lane;
  }, 8 * kBrickGrain);
  h->slab_order = order;
  if (order == HLB_ORDER_AUTO) {
    // median slab distance from a brick to its y neighbour in TILE order
    std::vector<int64_t> first((size_t)NBr + 1, 0);
    for (int64_t k = 0; k < NBr; ++k) {
      int n = 0;
      for (int x = 0; x < 8; ++x) n += fmAll[(size_t)k * 8 + x] != 0;
      first[(size_t)k + 1] = first[(size_t)k] + n;
    }
    std::vector<int64_t> dist;
    for (int64_t k = 0; k < NBr; ++k) {
      const int64_t t = brickTile[(size_t)k], ty = (t / ntz) % nty;
      if (ty + 1 >= nty) continue;
      const int32_t nb = brickOf[(size_t)(t + ntz)];
      if (nb >= 0) dist.push_back(first[(size_t)nb] - first[(size_t)k]);
    }
    int64_t median = 0;
    if (!dist.empty()) {
      std::nth_element(dist.begin(), dist.begin() + dist.size() / 2, dist.end());
      median = dist[dist.size() / 2];
    }
    h->slab_order = median > kL2WindowSlabs ? HLB_ORDER_LAYER : HLB_ORDER_TILE;
  }
  const bool layer = h->slab_order == HLB_ORDER_LAYER;
  // active slabs, their masks and compact bases
  std::vector<int32_t> slabOf((size_t)NBr * 8, -1);
  h->h_slab.clear();
  h->h_sbase.clear();
  h->h_fmask.clear();
  int64_t next = 0;
  for (int64_t i = 0; i < NBr * 8; ++i) {
    const int64_t k = layer ? i % NBr : i / 8;
    const int x = (int)(layer ? i / NBr : i % 8);
    const uint64_t fm = fmAll[(size_t)k * 8 + x];
    if (fm == 0) continue;
    next = round_up(next, kSlabAlign);
    slabOf[(size_t)k * 8 + x] = (int32_t)h->h_slab.size();
    h->h_slab.push_back((int32_t)(k * 8 + x));
    h->h_sbase.push_back((int32_t)next);
    h->h_fmask.push_back(fm);
    next += __builtin_popcountll(fm);
  }
  h->nslab = (int64_t)h->h_slab.size();
  h->S = round_up(std::max<int64_t>(next, 1), 64);
  h->perm.assign((size_t)h->S, -1);
  h->inv.assign((size_t)N, -1);
  h->h_rec.assign((size_t)std::max<int64_t>(h->nslab, 1), SlabRec{});
  // the slab at layer x + dx of the brick at (dy, dz) from brick k, or -1
  auto reach = [&](int64_t k, int x, int dx, int dy, int dz) -> int32_t {
    const int xx = x + dx;
    const int bx = xx < 0 ? -1 : (xx > 7 ? 1 : 0);
    const int64_t t = brickTile[k];
    const int64_t tx = t / (nty * ntz) + bx, ty = (t / ntz) % nty + dy, tz = t % ntz + dz;
    if (tx < 0 || ty < 0 || tz < 0 || tx >= ntx || ty >= nty || tz >= ntz) return -1;
    const int32_t nb = brickOf[tile_of(tx, ty, tz)];
    return nb < 0 ? -1 : slabOf[(size_t)nb * 8 + (xx & 7)];
  };
  // per slab its boundary and iolet sites, then where their numbering starts
  std::vector<int32_t> firstB((size_t)h->nslab + 1, 0), firstI((size_t)h->nslab + 1, 0);
  constexpr int64_t kSlabGrain = kGrain / kSlab;
  parallel_ranges(h->nslab, [&](int, int64_t lo, int64_t hi) {
    for (int64_t r = lo; r < hi; ++r) {
      const int32_t* sites = &at[(size_t)h->h_slab[r] * kSlab];
      for (int lane = 0; lane < kSlab; ++lane) {
        if (sites[lane] >= L.off[1]) firstB[(size_t)r + 1]++;
        if (sites[lane] >= L.off[2]) firstI[(size_t)r + 1]++;
      }
    }
  }, kSlabGrain);
  for (int64_t r = 0; r < h->nslab; ++r) {
    firstB[(size_t)r + 1] += firstB[(size_t)r];
    firstI[(size_t)r + 1] += firstI[(size_t)r];
  }
  h->bsite.resize((size_t)firstB.back());
  h->isite.resize((size_t)firstI.back());
  // fluid neighbours of all sites: as many as plain links, unless wall or iolet
  // links lead to fluid sites (counted here, 64 sites at a time, because the same
  // test per link takes 7% of hlb_create)
  std::atomic<int64_t> neighbours{0};
  parallel_ranges(h->nslab, [&](int, int64_t lo, int64_t hi) {
    int64_t count = 0;
    for (int64_t r = lo; r < hi; ++r) {
      const int64_t k = h->h_slab[r] >> 3;
      const int x = h->h_slab[r] & 7;
      SlabRec& R = h->h_rec[r];
      std::memset(&R, 0, sizeof R);
      R.sid = h->h_slab[r];
      R.bbase = firstB[(size_t)r];
      for (int dx = -1; dx <= 1; ++dx)
        for (int dy = -1; dy <= 1; ++dy)
          for (int dz = -1; dz <= 1; ++dz) {
            if (dx != 0 && dy != 0 && dz != 0) continue;  // no such link in D3Q19
            const int e = reach_entry(dx, dy, dz);
            const int32_t q = reach(k, x, dx, dy, dz);
            R.fm[e] = q < 0 ? 0 : h->h_fmask[q];
            R.base[e] = q < 0 ? 0 : h->h_sbase[q];
          }
      int32_t nb = firstB[(size_t)r], ni = firstI[(size_t)r];
      uint32_t slot = (uint32_t)h->h_sbase[r];
      for (int lane = 0; lane < kSlab; ++lane) {
        const int32_t site = at[(size_t)h->h_slab[r] * kSlab + lane];
        if (site < 0) continue;
        h->perm[slot] = site;
        h->inv[site] = (int32_t)slot;
        ++slot;
        if (site >= L.off[1]) {
          R.bmask |= 1ull << lane;
          h->bsite[(size_t)nb++] = site;
        }
        if (site >= L.off[2]) h->isite[(size_t)ni++] = site;
      }
      count += fluid_neighbours(R);
    }
    neighbours.fetch_add(count, std::memory_order_relaxed);
  }, kSlabGrain);
  if (neighbours.load() != (Q - 1) * N - L.links) mark_inner_links(h->L);
  h->NB = (int64_t)h->bsite.size();
  h->NI = (int64_t)h->isite.size();
  h->SB = round_up(std::max<int64_t>(h->NB, 1), 64);
  h->SI = round_up(std::max<int64_t>(h->NI, 1), 64);
}

// Ladd profile factors s = 1 - r^2/a^2 at each velocity link's half-way
// point (LaddIoletDelegate.h:66-69, InOutLetParabolicVelocity.cc:30-45).  The
// reference stops with std::exit(16) when a half-way point lies outside the
// iolet radius; here hlb_create fails with HLB_ERANGE.
int ladd_factors(hlb_lattice* h) {
  const HostLattice& L = h->L;
  const int64_t SI = h->SI;
  std::vector<double>& s = h->h_ladd_s;
  s.assign((size_t)36 * SI, 0.0);
  for (int64_t i = 0; i < h->NI; ++i) {
    const int64_t k = h->isite[i];
    const int c = L.collision_class(k);
    const bool inletSide = (c == 2 || c == 4);
    const int bc = inletSide ? h->params.inlet_bc : h->params.outlet_bc;
    if (bc != HLB_IOLET_LADD) continue;
    const HostIolet& io = h->iolets[side_iolet(h, k)];
    for (int d = 1; d < Q; ++d) {
      if (!((L.iolet[k] >> (d - 1)) & 1u)) continue;
      // LaddIoletDelegate::StreamLink: the velocity at the link's half-way point
      const double x[3] = {(double)L.coords[3 * k] + 0.5 * CX[d], (double)L.coords[3 * k + 1] + 0.5 * CY[d],
                           (double)L.coords[3 * k + 2] + 0.5 * CZ[d]};
      double f1 = 0.0, f2 = 0.0;
      const int rc = velocity_factors(io, x, f1, f2);
      if (rc != HLB_OK) return rc;
      s[(size_t)(d - 1) * SI + i] = f1;
      s[(size_t)(18 + d - 1) * SI + i] = f2;
    }
  }
  return HLB_OK;
}

// Windkessel bookkeeping: coupling direction, centre site and coupling sites
// of every Windkessel iolet.  A site couples when it has an iolet link in
// direction INV[dirs0] (the streamers call DoPreStreamCoupling for the link
// whose unstreamed direction is dirs0, NashZerothOrderPressureDelegate.h:46-52).
void windkessel_setup(hlb_lattice* h) {
  const HostLattice& L = h->L;
  const int nio = (int)h->iolets.size();
  h->wk_host.assign(std::max(1, nio), WkIolet{});
  h->wk_list.clear();
  std::vector<std::vector<int32_t>> lists(nio);
  std::vector<int32_t> iolIndex(L.N, -1);
  for (int64_t i = 0; i < h->NI; ++i) iolIndex[h->isite[i]] = (int32_t)i;
  for (int g = 0; g < nio; ++g) {
    HostIolet& io = h->iolets[g];
    io.dirs0 = direction_closest_to(io.n);
    io.centre = -1;
    for (int64_t k = 0; k < L.N && io.IsWK(); ++k) {
      bool in = true;
      for (int a = 0; a < 3; ++a) {
        const double c = (double)L.coords[3 * k + a];
        in = in && (c >= io.d.position[a] - 1.0) && (c <= io.d.position[a] + 1.0);
      }
      if (in) {
        io.centre = k;
        break;
      }
    }
  }
  for (int64_t k = L.off[2]; k < L.N; ++k) {  // reference order
    const int g = side_iolet(h, k);
    HostIolet& io = h->iolets[g];
    if (!io.IsWK()) continue;
    const int link = INV[io.dirs0];
    if (link == 0 || !((L.iolet[k] >> (link - 1)) & 1u)) continue;
    lists[g].push_back(iolIndex[k]);
    if (k == io.centre) io.centreCoupled = true;
  }
  for (int g = 0; g < nio; ++g) {
    const HostIolet& io = h->iolets[g];
    WkIolet& w = h->wk_host[g];
    w.density = w.densityNew = 1.0;
    w.flowRate = w.flowRateOld = w.flowRateNew = w.siteCount = 0.0;
    w.area = io.d.area;
    w.resistance = io.d.resistance;
    w.r_c = io.d.r_c;
    w.r_p = io.d.r_p;
    w.capacitance = io.d.capacitance;
    w.kind = io.d.kind;
    w.centre_coupled = io.centreCoupled ? 1 : 0;
    w.list_begin = (int32_t)h->wk_list.size();
    h->wk_list.insert(h->wk_list.end(), lists[g].begin(), lists[g].end());
    w.list_end = (int32_t)h->wk_list.size();
    if (io.IsWK()) h->any_wk = true;
  }
}

// Guo-Zheng-Shi wall links (GuoZhengShiDelegate.h:123-294): which wall links
// take a GZS value and which branch they follow (the rest bounce back), the
// sites whose pre-collision f the link kernel reads, numbered in slot order,
// and their per-slab masks.
int gzs_setup(hlb_lattice* h) {
  const HostLattice& L = h->L;
  h->gz_links_host.clear();
  h->h_pmask.clear();
  h->h_pbase.clear();
  h->h_bgz.assign((size_t)h->SB, 0);
  h->h_bgzbase.assign((size_t)h->SB, 0);
  h->NP = 0;
  if (h->params.wall_bc != HLB_WALL_GZS) return HLB_OK;
  struct Pending {
    int64_t k, nb;
    int d, mode, gi;
    float q;
    double s, s2;
  };
  std::vector<Pending> pend;
  std::vector<uint8_t> needP(L.N, 0);
  for (int64_t b = 0; b < h->NB; ++b) {
    const int64_t k = h->bsite[b];
    const uint32_t wm = L.wall[k], im = L.iolet[k];
    h->h_bgzbase[b] = (int32_t)pend.size();
    for (int d = 1; d < Q; ++d) {
      if (!((wm >> (d - 1)) & 1u)) continue;
      const int i = INV[d];
      const float q = L.q[k * 18 + d - 1];
      int mode = 1, gi = -1;
      int64_t nb = -1;
      double sfac = 0.0, sfac2 = 0.0;
      if ((double)q < 0.75) {
        if ((im >> (i - 1)) & 1u) {
          gi = side_iolet(h, k);
          const HostIolet& io = h->iolets[gi];
          if (!io.IsVelocity()) continue;  // bounce-back
          const double x[3] = {(double)L.coords[3 * k] + CX[i], (double)L.coords[3 * k + 1] + CY[i],
                               (double)L.coords[3 * k + 2] + CZ[i]};
          const int rc = velocity_factors(io, x, sfac, sfac2);
          if (rc != HLB_OK) return rc;
          mode = 3;
        } else if ((wm >> (i - 1)) & 1u) {
          continue;  // bounce-back
        } else {
          nb = L.site_at(L.coords[3 * k] + CX[i], L.coords[3 * k + 1] + CY[i], L.coords[3 * k + 2] + CZ[i]);
          if (nb < 0) return fail(HLB_EGEOMETRY, "hlb_create: GZS needs a fluid site beyond a wall link's opposite");
          mode = 2;
          needP[nb] = 1;
        }
      }
      needP[k] = 1;
      h->h_bgz[b] |= 1u << (d - 1);
      pend.push_back({k, nb, d, mode, gi, q, sfac, sfac2});
    }
  }
  std::vector<int32_t> pidx(L.N, -1);
  for (size_t r = 0; r < h->h_slab.size(); ++r) {
    const uint64_t fm = h->h_fmask[r];
    uint64_t pm = 0;
    h->h_pbase.push_back((int32_t)h->NP);
    int32_t slot = h->h_sbase[r];
    for (int lane = 0; lane < kSlab; ++lane) {
      if (!((fm >> lane) & 1u)) continue;
      const int32_t k = h->perm[slot++];
      if (!needP[k]) continue;
      pm |= 1ull << lane;
      pidx[k] = (int32_t)h->NP++;
    }
    h->h_pmask.push_back(pm);
  }
  for (const Pending& p : pend)
    h->gz_links_host.push_back(GzsLink{pidx[p.k], p.nb >= 0 ? pidx[p.nb] : -1, p.d, p.mode, p.gi, p.q, p.s, p.s2});
  h->SP = round_up(std::max<int64_t>(h->NP, 1), 64);
  return HLB_OK;
}

// The sponge's vTau planes (double for the FP64 step and the stress caches,
// float as well for the FP32-shifted step); nothing without a sponge.
int upload_sponge(hlb_lattice* h) {
  if (h->sponge_life <= 0 || h->h_vtau.empty()) return HLB_OK;
  const size_t S = (size_t)h->S;
  HLB_CHECK(h->vtau64.alloc(S));
  HLB_CHECK(copy_now(h->vtau64.p, h->h_vtau.data(), sizeof(double) * S, hipMemcpyHostToDevice, h->stream));
  if (h->fp32()) {
    std::vector<float> v(S);
    for (size_t i = 0; i < S; ++i) v[i] = (float)h->h_vtau[i];
    HLB_CHECK(h->vtau32.alloc(S));
    HLB_CHECK(copy_now(h->vtau32.p, v.data(), sizeof(float) * S, hipMemcpyHostToDevice, h->stream));
  }
  return HLB_OK;
}

int upload_lattice(hlb_lattice* h) {
  const HostLattice& L = h->L;
  const int64_t N = L.N, S = h->S, SB = h->SB, SI = h->SI, NB = h->NB;
  DevPack pack;
  // the two distribution sets are one allocation, the field arrays another
  if (h->fp32()) {
    HLB_CHECK(h->a_mem.alloc(sizeof(float) * 2 * Q * S));
    for (int c = 0; c < 2; ++c) h->A32[c].view(h->a_mem.p + sizeof(float) * Q * S * c, (size_t)Q * S);
    pack.add(h->G32, (const float*)nullptr, (size_t)Q * SI);
    pack.add(h->feq32, (const float*)nullptr, (size_t)Q);
  } else {
    HLB_CHECK(h->a_mem.alloc(sizeof(double) * 2 * Q * S));
    for (int c = 0; c < 2; ++c) h->A[c].view(h->a_mem.p + sizeof(double) * Q * S * c, (size_t)Q * S);
    pack.add(h->G, (const double*)nullptr, (size_t)Q * SI);
  }
  HLB_CHECK(hipMemsetAsync(h->a_mem.p, 0, h->a_mem.n, h->stream));
  // Holes are never written: keep the field arrays defined there.
  HLB_CHECK(h->fields_mem.alloc(sizeof(double) * 5 * S));
  HLB_CHECK(hipMemsetAsync(h->fields_mem.p, 0, h->fields_mem.n, h->stream));
  h->rho.view(h->fields_mem.p, (size_t)S);
  h->u.view(h->fields_mem.p + sizeof(double) * S, (size_t)3 * S);
  h->wss.view(h->fields_mem.p + sizeof(double) * 4 * S, (size_t)S);
  pack.add(h->feq_vals, (const double*)nullptr, (size_t)Q);

  // Guo-Zheng-Shi tables.
  {
    const int rc = gzs_setup(h);
    if (rc != HLB_OK) return rc;
    if (!h->gz_links_host.empty()) {
      const size_t nl = h->gz_links_host.size();
      pack.add(h->gz_links, h->gz_links_host);
      pack.add(h->pmask, h->h_pmask);
      pack.add(h->pbase, h->h_pbase);
      pack.add(h->bgz, reinterpret_cast<const uint32_t*>(h->h_bgz.data()), (size_t)SB);
      pack.add(h->bgzbase, h->h_bgzbase.data(), (size_t)SB);
      if (h->fp32()) {
        HLB_CHECK(h->P32.alloc((size_t)Q * h->SP));
        HLB_CHECK(h->GW32.alloc(nl));
      } else {
        HLB_CHECK(h->P64.alloc((size_t)Q * h->SP));
        HLB_CHECK(h->GW64.alloc(nl));
      }
    }
  }
  // Slab records and the site -> slot index.
  pack.add(h->rec, h->h_rec);
  pack.add(h->dinv, h->inv.data(), h->inv.size());
  // Boundary arrays in device order.
  std::vector<BndRec> rec(SB, BndRec{0, 0, 0, 0});
  std::vector<float> q((size_t)18 * SB, 0.0f), nr((size_t)3 * SB, 0.0f);
  std::vector<uint32_t> inner(h->inner_links() ? (size_t)SB : 0, 0);
  {
    std::vector<int32_t> iolIndex(N, -1);
    for (int64_t i = 0; i < h->NI; ++i) iolIndex[h->isite[i]] = (int32_t)i;
    parallel_ranges(NB, [&](int, int64_t lo, int64_t hi) {
      for (int64_t b = lo; b < hi; ++b) {
        const int64_t k = h->bsite[b];
        BndRec& R = rec[b];
        const uint32_t wm = L.wall[k];
        R.iolet = L.iolet[k];
        if (wm != 0) R.far |= 1u << 31;
        if (!inner.empty() && (inner[(size_t)b] = L.inner[(size_t)k]) != 0) R.far |= kInnerLinks;
        // BouzidiFirdaousLallemandDelegate.h:44-93: a wall link whose opposite is
        // no wall interpolates, with the site's own opposite value from q = 1/2 on
        for (int j = 1; j < Q && h->params.wall_bc == HLB_WALL_BFL; ++j) {
          const int ib = INV[j];
          if (!((wm >> (ib - 1)) & 1u) || ((wm >> (j - 1)) & 1u)) continue;
          (L.q[k * 18 + ib - 1] < 0.5f ? R.near : R.far) |= 1u << (j - 1);
        }
        if (k >= L.off[2]) {
          R.near |= (uint32_t)side_iolet(h, k) << 18;
          R.ii = (uint32_t)iolIndex[k];
        }
        for (int d = 0; d < 18; ++d) q[(size_t)d * SB + b] = L.q[k * 18 + d];
        for (int a = 0; a < 3; ++a) nr[(size_t)a * SB + b] = L.nrm[k * 3 + a];
      }
    });
  }
  pack.add(h->bnd, rec);
  pack.add(h->bq, q);
  pack.add(h->bnrm, nr);
  pack.add(h->inner, inner);
  pack.add(h->ladd_s, h->h_ladd_s);
  // Per-iolet constants and what the per-step values are copied to.
  {
    const int nio = h->iolet_count();
    std::vector<float> nf((size_t)3 * nio, 0.0f);
    std::vector<double> nd((size_t)3 * nio, 0.0);
    for (size_t g = 0; g < h->iolets.size(); ++g)
      for (int a = 0; a < 3; ++a) {
        nf[3 * g + a] = h->iolets[g].nf[a];
        nd[3 * g + a] = h->iolets[g].n[a];
      }
    std::vector<uint32_t> bits(nio, 0u);
    for (size_t g = 0; g < h->iolets.size(); ++g)
      if (h->iolets[g].IsWK() && h->iolets[g].dirs0 != 0) bits[g] = 1u << (INV[h->iolets[g].dirs0] - 1);
    std::vector<int32_t> pos((size_t)std::max<int64_t>(1, SI), -1);
    for (size_t e = 0; e < h->wk_list.size(); ++e) pos[(size_t)h->wk_list[e]] = (int32_t)e;
    pack.add(h->io_nf, nf);
    pack.add(h->io_n, nd);
    pack.add(h->stage, (const double*)nullptr, (size_t)h->stage_doubles());
    pack.add(h->wk_bit, bits);
    pack.add(h->wk, h->wk_host);
    // the coupling terms, written by the step in the coupling order
    pack.add(h->wk_contrib, (const double*)nullptr, 2 * (size_t)h->wk_stride());
    pack.add(h->wk_pos, pos);
    HLB_CHECK(pack.commit(h->arena, h->stream));
    h->wk_refs_host.clear();
    for (size_t g = 0; g < h->iolets.size(); ++g)
      if (h->iolets[g].IsWK())
        h->wk_refs_host.push_back(WkRef{h->wk.p + g, h->rows(), h->wk_contrib.p, h->wk_stride(), (int32_t)g,
                                        (int32_t)h->row(), h->fp32() ? 0 : 1, 0});
    if (!h->wk_refs_host.empty()) {
      HLB_CHECK(h->wk_refs.alloc(h->wk_refs_host.size()));
      HLB_CHECK(copy_now(h->wk_refs.p, h->wk_refs_host.data(), sizeof(WkRef) * h->wk_refs_host.size(),
                         hipMemcpyHostToDevice, h->stream));
    }
  }
  {
    const int rc = upload_sponge(h);
    if (rc != HLB_OK) return rc;
  }
  HLB_CHECK(hipStreamSynchronize(h->stream));
  return HLB_OK;
}

}  // namespace

void advance_state(hlb_lattice* h, int64_t n) {
  if (n <= 0) return;
  h->cur = h->have_post ? (h->cur ^ (int)(n & 1)) : (h->cur ^ (int)((n - 1) & 1));
  h->have_post = true;
  h->t += n;
}

// Device state is created on first use so the host tables can be built and
// inspected on a machine without a GPU.
int ensure_device(hlb_lattice* h) {
  if (h->device_ready) return HLB_OK;
  if (!h->iolets_set) return fail(HLB_EINVAL, "the lattice has no iolets configured (hlb_set_iolets)");
  HLB_CHECK(hipGetDevice(&h->device));
  {
    // Test switch, read once per handle: the FP64 steady step takes its
    // general gather (the path of lattices above 2^28 slots) on any lattice.
    const char* force = std::getenv("HLB_FP64_GENERAL_GATHER");
    h->general_gather = force && force[0] == '1';
  }
  int rc = take_lane(h->device, (size_t)h->stage_doubles(), h->lane);
  if (rc != HLB_OK) return rc;
  h->use_lane();
  rc = upload_lattice(h);
  if (rc != HLB_OK) {
    // without a state the iolets, which size the staging, may still change
    (void)hipStreamSynchronize(h->stream);
    give_lane(h->lane);
    h->use_lane();
    return rc;
  }
  transfer_open();
  h->device_ready = true;
  return HLB_OK;
}

namespace {

int validate_core(const hlb_params& p, const char* who) {
  const std::string w(who);
  if (p.kernel < HLB_KERNEL_LBGK || p.kernel > HLB_KERNEL_LES) return fail(HLB_EINVAL, w + ": unknown kernel");
  if (p.wall_bc != HLB_WALL_SBB && p.wall_bc != HLB_WALL_BFL && p.wall_bc != HLB_WALL_GZS)
    return fail(HLB_EINVAL, w + ": unknown wall BC");
  if (p.wall_bc == HLB_WALL_GZS && p.kernel == HLB_KERNEL_LES)
    return fail(HLB_EINVAL, w + ": GZS walls are not defined with the LES kernel (the wall node has no LES tau)");
  for (int bc : {p.inlet_bc, p.outlet_bc})
    if (bc != HLB_IOLET_NASH && bc != HLB_IOLET_LADD) return fail(HLB_EINVAL, w + ": unknown iolet BC");
  if (p.precision != HLB_FP64 && p.precision != HLB_FP32_SHIFTED)
    return fail(HLB_EINVAL, w + ": unknown storage precision");
  if (!(p.tau > 0.5)) return fail(HLB_EINVAL, w + ": tau must exceed 1/2");
  if (p.slab_order < HLB_ORDER_AUTO || p.slab_order > HLB_ORDER_LAYER)
    return fail(HLB_EINVAL, w + ": unknown slab order");
  return HLB_OK;
}

int validate_iolets(const hlb_params& p, const hlb_iolet_desc* in, int nin, const hlb_iolet_desc* out, int nout,
                    const char* who) {
  const std::string w(who);
  for (int side = 0; side < 2; ++side) {
    const hlb_iolet_desc* v = side ? out : in;
    const int n = side ? nout : nin;
    const int bc = side ? p.outlet_bc : p.inlet_bc;
    if (n > 0 && !v) return fail(HLB_EINVAL, w + ": null iolet array");
    for (int i = 0; i < n; ++i) {
      const int k = v[i].kind;
      if (k < HLB_IOLET_COSINE || k > HLB_IOLET_WOMERSLEY) return fail(HLB_EINVAL, w + ": unknown iolet kind");
      if ((k == HLB_IOLET_WK2 || k == HLB_IOLET_WK3) && bc != HLB_IOLET_NASH)
        return fail(HLB_EINVAL, w + ": a Windkessel iolet needs the Nash pressure boundary");
      const bool vel = (k == HLB_IOLET_PARABOLIC || k == HLB_IOLET_FILEVEL || k == HLB_IOLET_WOMERSLEY);
      if (bc == HLB_IOLET_LADD && !vel)
        return fail(HLB_EINVAL, w + ": the Ladd boundary needs a velocity iolet (LaddIoletDelegate.h:51-53)");
      if (vel && !(v[i].radius > 0.0)) return fail(HLB_EINVAL, w + ": velocity iolet without radius");
      if (k == HLB_IOLET_FILEVEL && (!v[i].table || v[i].table_len <= 0))
        return fail(HLB_EINVAL, w + ": file velocity iolet without a table");
      if (k == HLB_IOLET_FILEPRES && (!v[i].table || v[i].table_len <= 0))
        return fail(HLB_EINVAL, w + ": file pressure iolet without a table");
      if (k == HLB_IOLET_WOMERSLEY && !(v[i].period != 0.0))
        return fail(HLB_EINVAL, w + ": Womersley iolet with zero period");
      if (k == HLB_IOLET_COSINE && !(v[i].period != 0.0)) return fail(HLB_EINVAL, w + ": cosine iolet with zero period");
    }
  }
  return HLB_OK;
}

// LbmParameters (LbmParameters.h:29-45) and the TRT / LES constants.  Once
// the lattice has a device state only tau and the TRT magic parameter may
// change (LbmParameters::Update).
int configure_params(hlb_lattice* h, const hlb_params& p, const char* who) {
  int rc = validate_core(p, who);
  if (rc != HLB_OK) return rc;
  const hlb_params& o = h->params;
  if (h->device_ready && (p.kernel != o.kernel || p.wall_bc != o.wall_bc || p.inlet_bc != o.inlet_bc ||
                          p.outlet_bc != o.outlet_bc || p.precision != o.precision))
    return fail(HLB_EINVAL, std::string(who) + ": only tau and trt_lambda can change once the lattice has a state");
  if (p.slab_order != HLB_ORDER_AUTO && p.slab_order != h->slab_order)
    return fail(HLB_EINVAL, std::string(who) + ": the slab order is fixed when the lattice is created");
  if (h->iolets_set && !h->device_ready) {
    std::vector<hlb_iolet_desc> in, out;
    for (int g = 0; g < (int)h->iolets.size(); ++g) (g < h->n_in ? in : out).push_back(h->iolets[g].d);
    for (auto* v : {&in, &out})
      for (size_t i = 0; i < v->size(); ++i) {
        const HostIolet& io = h->iolets[(v == &in ? 0 : h->n_in) + i];
        if (!io.table.empty()) {
          (*v)[i].table = io.table.data();
          (*v)[i].table_len = (int64_t)io.table.size();
        }
      }
    rc = validate_iolets(p, in.data(), (int)in.size(), out.data(), (int)out.size(), who);
    if (rc != HLB_OK) return rc;
  }
  h->params = p;
  h->params.slab_order = h->slab_order;
  if (!h->variant_chosen) h->variant = default_variant(distribution_bytes(h->S, h->fp32()), h->fp32());
  const double tau = p.tau;
  h->omega = -1.0 / tau;
  h->half_omega = 0.5 * h->omega;
  const double tau_minus = 0.5 + p.trt_lambda / (tau - 0.5);
  h->half_omega_minus = 0.5 * (-1.0 / tau_minus);
  {
    const double rho1 = 1.0, C_smag = 0.1;
    double k = 18.0 * 1.4142135623730950488016887242097;
    k = k * rho1;
    k = k * C_smag;
    k = k * C_smag;
    h->les_k = k;
  }
  if (h->iolets_set && !h->device_ready) return ladd_factors(h);
  return HLB_OK;
}

// BoundaryValues::BoundaryValues (src/lb/iolets/BoundaryValues.cc:20-81) and
// LBM::PrepareBoundaryObjects (src/lb/lb.hpp:119-143).
int configure_iolets(hlb_lattice* h, const hlb_iolet_desc* inlets, int n_inlets, const hlb_iolet_desc* outlets,
                     int n_outlets, const char* who) {
  const std::string w(who);
  if (h->device_ready) return fail(HLB_EINVAL, w + ": the iolets are fixed once the lattice has a state");
  if (n_inlets < 0 || n_outlets < 0) return fail(HLB_EINVAL, w + ": negative iolet count");
  if (n_inlets + n_outlets > kMaxIolets)
    return fail(HLB_EINVAL, w + ": at most " + std::to_string(kMaxIolets) + " iolets per lattice");
  int rc = validate_iolets(h->params, inlets, n_inlets, outlets, n_outlets, who);
  if (rc != HLB_OK) return rc;
  // Iolet ids on sites must name a configured iolet of the site's side.
  for (int64_t k = h->L.off[2]; k < h->L.N; ++k) {
    const int c = h->L.collision_class(k);
    const int lim = (c == 2 || c == 4) ? n_inlets : n_outlets;
    if (h->L.ioletId[k] < 0 || h->L.ioletId[k] >= lim)
      return fail(HLB_EINVAL, w + ": a site names iolet " + std::to_string(h->L.ioletId[k]) + " but only " +
                                  std::to_string(lim) + " are configured on its side");
  }
  h->iolets.clear();
  h->n_in = n_inlets;
  h->n_out = n_outlets;
  for (int side = 0; side < 2; ++side) {
    const hlb_iolet_desc* v = side ? outlets : inlets;
    const int n = side ? n_outlets : n_inlets;
    for (int i = 0; i < n; ++i) {
      HostIolet io;
      io.d = v[i];
      double nx = v[i].normal[0], ny = v[i].normal[1], nz = v[i].normal[2];
      if (!(nx == 0.0 && ny == 0.0 && nz == 0.0)) {
        const double mag = std::sqrt(nx * nx + ny * ny + nz * nz);
        nx /= mag;
        ny /= mag;
        nz /= mag;
      }
      io.n[0] = nx;
      io.n[1] = ny;
      io.n[2] = nz;
      io.nf[0] = (float)nx;
      io.nf[1] = (float)ny;
      io.nf[2] = (float)nz;
      if (v[i].kind == HLB_IOLET_FILEVEL || v[i].kind == HLB_IOLET_FILEPRES)
        io.table.assign(v[i].table, v[i].table + v[i].table_len);
      io.d.table = nullptr;
      h->iolets.push_back(std::move(io));
    }
  }
  // Every iolet learns the minimum density any iolet can impose.
  double minDensity = DBL_MAX;
  // GetDensityMin: cosine mean - amplitude (InOutLetCosine.h:55-58), file the
  // table's minimum pressure (InOutLetFile.h:48-51), others 1.
  for (const HostIolet& io : h->iolets)
    minDensity = std::min(minDensity, io.d.kind == HLB_IOLET_COSINE   ? io.d.density_mean - io.d.density_amp
                                      : io.d.kind == HLB_IOLET_FILEPRES ? io.d.density_min
                                                                        : 1.0);
  for (HostIolet& io : h->iolets) io.minSimDensity = minDensity;
  rc = ladd_factors(h);
  if (rc != HLB_OK) return rc;
  h->any_wk = false;
  windkessel_setup(h);
  h->iolets_set = true;
  return HLB_OK;
}

}  // namespace

// The member record of an FP32 handle for a launch sequence starting now.
Member32 member_record(const hlb_lattice* h, int props_at) {
  Member32 m{};
  m.A[0] = h->A32[0].p;
  m.A[1] = h->A32[1].p;
  m.F = h->F32.p;
  m.bt = h->tables();
  m.gz = h->gz_tables();
  m.P = h->P32.p;
  m.GW = h->GW32.p;
  m.bnd = h->bnd.p;
  m.bq = h->bq.p;
  m.bnrm = h->bnrm.p;
  m.G = h->G32.p;
  m.ladd_s = h->ladd_s.p;
  m.ladd_s2 = h->ladd_s.p ? h->ladd_s.p + (size_t)18 * h->SI : nullptr;
  m.rho = h->rho.p;
  m.u = h->u.p;
  m.wss = h->wss.p;
  m.io_nf = h->io_nf.p;
  m.io_n = h->io_n.p;
  m.io_dens = h->rows();
  m.io_vmax = m.io_dens + h->iolet_count();
  m.io_vmax2 = m.io_dens + 2 * h->iolet_count();
  m.wk_bit = h->wk_bit.p;
  m.wk_pos = h->wk_pos.p;
  m.wk_contrib = h->wk_contrib.p;
  m.wk_stride = h->wk_stride();
  m.N = h->L.N;
  m.S = h->S;
  m.SB = h->SB;
  m.SI = h->SI;
  m.row = (int32_t)h->row();
  m.n_in = h->n_in;
  m.kernel = h->params.kernel;
  m.inlet_bc = h->params.inlet_bc;
  m.outlet_bc = h->params.outlet_bc;
  m.cur0 = h->cur;
  m.first0 = h->have_post ? 0 : 1;
  m.props_at = props_at;
  m.wg_begin = 0;
  m.tau = (float)h->params.tau;
  m.omega = (float)h->omega;
  m.half_omega = (float)h->half_omega;
  m.half_omega_minus = (float)h->half_omega_minus;
  m.les_k = (float)h->les_k;
  m.vtau = h->sponge_life > 0 ? h->vtau32.p : nullptr;
  m.sp_t = m.io_dens + 3 * h->iolet_count();
  m.sp_half = (double)(h->sponge_life / 2);
  m.sp_life = (double)h->sponge_life;
  return m;
}

namespace {

uint32_t member_grid(int64_t nslab, int variant) {
  const LaunchShape l = launch_shape(variant, true);
  const int64_t per = shape_slabs(l);
  return shape_grid(l, (nslab + per - 1) / per);
}

// Writes the member record through the head of the pinned staging; the caller
// has synchronised the stream, so the staging is free.
int upload_member(hlb_lattice* h, int props_at) {
  h->staging_idle = false;
  const Member32 m = member_record(h, props_at);
  std::memcpy(h->h_stage, &m, sizeof m);
  HLB_CHECK(hipMemcpyAsync(h->stage.p, h->h_stage, sizeof m, hipMemcpyHostToDevice, h->stream));
  return HLB_OK;
}

// Forms the rows of steps t .. t+n-1 in the pinned staging: per iolet the ghost
// density and the two speed factors, then the sponge's time.
int form_rows(hlb_lattice* h, int64_t t, int64_t n) {
  h->staging_idle = false;
  const int64_t nio = h->iolet_count(), row = h->row();
  for (int64_t s = 0; s < n; ++s) {
    double* r = h->h_stage + kStageHead + s * row;
    const int rc = iolet_values(h, t + s, r, r + nio, r + 2 * nio);
    if (rc != HLB_OK) return rc;
    // LBGKLESSpongeLayer::CalculateTau reads the 1-indexed step; past the
    // lifetime the Smagorinsky time applies alone (-1).
    r[3 * nio] = t + s < h->sponge_life ? (double)(t + s) : -1.0;
  }
  return HLB_OK;
}

}  // namespace

int stage_iolet_values(hlb_lattice* h, int64_t t, int64_t n, hipStream_t stream) {
  const int rc = form_rows(h, t, n);
  if (rc != HLB_OK) return rc;
  HLB_CHECK(hipMemcpyAsync(h->rows(), h->h_stage + kStageHead, sizeof(double) * n * h->row(), hipMemcpyHostToDevice,
                           stream));
  return HLB_OK;
}

namespace {

// Everything a sequence of n steps reads from the host, in one copy: the
// member record (FP32 form) and the rows behind it (no copy for rows read in
// place).  The caller has synchronised the stream.
int stage_sequence(hlb_lattice* h, int64_t n, bool props_last) {
  if (h->rows_in_place(n)) return form_rows(h, h->t, n);
  if (!h->fp32()) return stage_iolet_values(h, h->t, n, h->stream);
  const int rc = form_rows(h, h->t, n);
  if (rc != HLB_OK) return rc;
  const Member32 m = member_record(h, props_last ? (int)(n - 1) : -1);
  std::memcpy(h->h_stage, &m, sizeof m);
  HLB_CHECK(hipMemcpyAsync(h->stage.p, h->h_stage, sizeof(double) * (kStageHead + n * h->row()), hipMemcpyHostToDevice,
                           h->stream));
  return HLB_OK;
}

// Enqueues the launches of n steps whose iolet values (and, in the FP32
// form, member record) are staged: kernel launches only, so the sequence can
// be captured into a graph.
int enqueue_steps(hlb_lattice* h, int64_t n, bool props_last) {
  if (n <= 0) return HLB_OK;
  const int nwk = (int)h->wk_refs_host.size();
  const int variant = h->launch_variant();
  const WkLaunch wk = wk_launch(h->wk_refs.p, nwk, n);
  HLB_CHECK(launch_wk_start(h->wk_refs.p, nwk, h->stream));
  if (h->fp32()) {
    const uint32_t grid = member_grid(h->nslab, variant);
    for (int64_t s = 0; s < n; ++s) {
      HLB_CHECK(launch_step_fp32(h->member(), nullptr, grid, (int)s, wk, variant, h->inner_links(), h->stream));
      HLB_CHECK(launch_gzs_fp32(h->member(), h->gz_links.p, (int)h->gz_links_host.size(), (int)s, h->stream));
    }
    HLB_CHECK(launch_wk_flush(h->wk_refs.p, nwk, (int)(n - 1), h->stream));
    advance_state(h, n);
    return HLB_OK;
  }
  const double* rows = h->rows_in_place(n) ? h->h_stage + kStageHead : h->rows();
  for (int64_t s = 0; s < n; ++s) {
    const bool first = !h->have_post;
    const bool props = props_last && (s == n - 1);
    const double* ain = first ? h->F.p : h->A[h->cur].p;
    double* aout = first ? h->A[h->cur].p : h->A[h->cur ^ 1].p;
    StepArgs a = make_args(h, ain, aout);
    step_rows(h, a, rows, s);
    a.step = (int32_t)s;
    a.wk = wk;
    a.wk_contrib = h->wk_contrib.p + (s & 1) * h->wk_stride();
    HLB_CHECK(launch_step_fp64(a, h->params.kernel, first, props, variant, h->stream));
    HLB_CHECK(launch_gzs_fp64(a, h->params.kernel, h->gz_links.p, (int)h->gz_links_host.size(), a.io_vmax,
                              h->GW64.p, h->stream));
    if (!first) h->cur ^= 1;
    h->have_post = true;
  }
  HLB_CHECK(launch_wk_flush(h->wk_refs.p, nwk, (int)(n - 1), h->stream));
  h->t += n;
  return HLB_OK;
}

constexpr size_t kMaxStepGraphs = 8;  // replayable sequences kept per handle

// The captured sequence of the next n steps in the handle's current state,
// or nullptr.
const hlb_lattice::StepGraph* find_graph(const hlb_lattice* h, int64_t n, bool props_last) {
  const int first = h->fp32() ? 0 : (h->have_post ? 0 : 1);
  const int cur = h->fp32() ? 0 : h->cur;
  const int props = props_last ? 1 : 0;
  for (const auto& g : h->graphs)
    if (g.n == n && g.props == props && g.first == first && g.cur == cur && g.variant == h->launch_variant()) return &g;
  return nullptr;
}

// Makes sure the next n-step sequence has a graph: records the eager
// launches of enqueue_steps into one (nothing runs, the state does not
// advance).  At most kMaxStepGraphs are kept; the oldest goes first.
int prepare_graph(hlb_lattice* h, int64_t n, bool props_last) {
  if (find_graph(h, n, props_last)) return HLB_OK;
  const int first = h->fp32() ? 0 : (h->have_post ? 0 : 1);
  const int cur = h->fp32() ? 0 : h->cur;
  const int cur0 = h->cur;
  const bool have_post0 = h->have_post;
  const int64_t t0 = h->t;
  HLB_CHECK(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
  const int rc = enqueue_steps(h, n, props_last);
  hipGraph_t graph = nullptr;
  const hipError_t end = hipStreamEndCapture(h->stream, &graph);
  h->cur = cur0;
  h->have_post = have_post0;
  h->t = t0;
  if (rc != HLB_OK) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  HLB_CHECK(end);
  hipGraphExec_t exec = nullptr;
  const hipError_t inst = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
  (void)hipGraphDestroy(graph);
  HLB_CHECK(inst);
  if (h->graphs.size() >= kMaxStepGraphs) {
    // the oldest graph may still be running on the stream
    HLB_CHECK(hipStreamSynchronize(h->stream));
    (void)hipGraphExecDestroy(h->graphs.front().exec);
    h->graphs.erase(h->graphs.begin());
  }
  h->graphs.push_back({n, props_last ? 1 : 0, first, cur, h->launch_variant(), exec});
  return HLB_OK;
}

// Replays the prepared graph of the next n steps and advances the state.
int replay_graph(hlb_lattice* h, int64_t n, bool props_last) {
  const hlb_lattice::StepGraph* g = find_graph(h, n, props_last);
  if (!g) return fail(HLB_EINVAL, "internal: no graph prepared for this step sequence");
  HLB_CHECK(hipGraphLaunch(g->exec, h->stream));
  advance_state(h, n);
  return HLB_OK;
}

// Launches n staged steps, from a graph (captured on first use) or eagerly;
// the handle's state advances by n steps.
int launch_steps(hlb_lattice* h, int64_t n, bool props_last) {
  if (n <= 0) return HLB_OK;
  if (!h->use_graph || !h->replays(n)) return enqueue_steps(h, n, props_last);
  const int rc = prepare_graph(h, n, props_last);
  if (rc != HLB_OK) return rc;
  return replay_graph(h, n, props_last);
}

int run_steps(hlb_lattice* h, int64_t nsteps, uint32_t flags) {
  if (nsteps < 0) return fail(HLB_EINVAL, "hlb_step: negative step count");
  if (!h->f_valid) return fail(HLB_EINVAL, "hlb_step: no initial condition (call hlb_init_equilibrium or hlb_upload_f)");
  int64_t done = 0;
  while (done < nsteps) {
    const int64_t chunk = std::min<int64_t>(kChunk, nsteps - done);
    // The staging buffers are reused per chunk: wait for the launches that
    // read the previous chunk's values.
    if (!h->staging_idle) HLB_CHECK(hipStreamSynchronize(h->stream));
    const bool props_last = (flags & HLB_STEP_PROPERTIES) && done + chunk == nsteps;
    int rc = stage_sequence(h, chunk, props_last);
    if (rc != HLB_OK) return rc;
    rc = launch_steps(h, chunk, props_last);
    if (rc != HLB_OK) return rc;
    done += chunk;
  }
  return HLB_OK;
}

// Pre-collision f entering step t into F (device order, SoA).
int materialise_f(hlb_lattice* h) {
  if (!h->have_post) return HLB_OK;  // F already holds it
  if (h->fp32()) {
    if (!h->F32.p) HLB_CHECK(h->F32.alloc((size_t)Q * h->S));
    HLB_CHECK(hipStreamSynchronize(h->stream));
    int rc = upload_member(h, -1);
    if (rc != HLB_OK) return rc;
    HLB_CHECK(launch_gather_fp32(h->member(), h->nslab, h->F32.p, h->stream));
    return HLB_OK;
  }
  if (!h->F.p) HLB_CHECK(h->F.alloc((size_t)Q * h->S));
  StepArgs a = make_args(h, h->A[h->cur].p, nullptr);
  HLB_CHECK(launch_gather_fp64(a, h->F.p, h->S, h->stream));
  return HLB_OK;
}

}  // namespace
}  // namespace hlb

using namespace hlb;

extern "C" const char* hlb_last_error(void) { return last_error().c_str(); }

extern "C" int hlb_create(const hlb_geometry* geom, const hlb_params* params, const hlb_iolet_desc* inlets,
                          int n_inlets, const hlb_iolet_desc* outlets, int n_outlets, hlb_handle* out) {
  try {
    if (!geom || !out) return fail(HLB_EINVAL, "hlb_create: null argument");
    hlb_params p{};
    p.kernel = HLB_KERNEL_LBGK;
    p.wall_bc = HLB_WALL_SBB;
    p.inlet_bc = p.outlet_bc = HLB_IOLET_NASH;
    p.precision = HLB_FP64;
    p.tau = 1.0;
    p.trt_lambda = 3.0 / 16.0;
    if (params) p = *params;
    int rc = validate_core(p, "hlb_create");
    if (rc != HLB_OK) return rc;
    if (params) {
      if (n_inlets < 0 || n_outlets < 0) return fail(HLB_EINVAL, "hlb_create: negative iolet count");
      rc = validate_iolets(p, inlets, n_inlets, outlets, n_outlets, "hlb_create");
      if (rc != HLB_OK) return rc;
    }
    auto h = std::make_unique<hlb_lattice>();
    rc = build_lattice(*geom, h->L);
    if (rc != HLB_OK) return rc;
    h->params.precision = p.precision;  // the automatic order goes by the size of the distributions
    device_order(h.get(), p.slab_order);
    if (h->S > (int64_t(1) << 29))
      return fail(HLB_EINVAL, "hlb_create: the geometry needs " + std::to_string(h->S) +
                                  " device slots (occupied 8^3 tiles x 512), more than 2^29");
    rc = configure_params(h.get(), p, "hlb_create");
    if (rc != HLB_OK) return rc;
    if (params) {
      rc = configure_iolets(h.get(), inlets, n_inlets, outlets, n_outlets, "hlb_create");
      if (rc != HLB_OK) return rc;
    }
    *out = h.release();
    return HLB_OK;
  } catch (const std::bad_alloc&) {
    return fail(HLB_EINVAL, "hlb_create: out of host memory");
  }
}

namespace hlb {
namespace {

// LBGKLESSpongeLayer::InitState (src/lb/kernels/LBGKLESSpongeLayer.h:87-116)
// in device slot order: per site, the product over outlets within `width` of
// 1 + (ratio - 1)(dist / width - 1)^2, then vTau = product (tau0 - 1/2) + 1/2.
// The site-to-outlet vector is the reference's LatticeVector minus
// LatticePosition, which Vector3D<int64>::operator- (src/util/Vector3D.h:
// 396-399) evaluates after truncating the outlet position to int64 through
// the converting constructor (:237-243); its squared length is an int64 sum
// (:342-345).  Padding slots hold tau0.
void compute_sponge(hlb_lattice* h) {
  const HostLattice& L = h->L;
  const double width = h->sponge_width, widthSq = width * width, ratio = h->sponge_ratio;
  const double tau0 = h->params.tau;
  h->h_vtau.assign((size_t)h->S, tau0);
  for (int64_t slot = 0; slot < h->S; ++slot) {
    const int32_t k = h->perm[(size_t)slot];
    if (k < 0) continue;
    double vRatioTot = 1.0;
    for (int o = 0; o < h->n_out; ++o) {
      const double* pos = h->iolets[(size_t)(h->n_in + o)].d.position;
      const int64_t dx = (int64_t)L.coords[3 * (size_t)k] - (int64_t)pos[0];
      const int64_t dy = (int64_t)L.coords[3 * (size_t)k + 1] - (int64_t)pos[1];
      const int64_t dz = (int64_t)L.coords[3 * (size_t)k + 2] - (int64_t)pos[2];
      const double distSq = (double)(dx * dx + dy * dy + dz * dz);
      const double dist = std::sqrt(distSq);
      if (distSq <= widthSq) vRatioTot *= 1.0 + (ratio - 1.0) * (dist / width - 1.0) * (dist / width - 1.0);
    }
    h->h_vtau[(size_t)slot] = vRatioTot * (tau0 - 0.5) + 0.5;
  }
}

// Recomputes and uploads the sponge after a change of tau or outlets.
int refresh_sponge(hlb_lattice* h) {
  if (h->sponge_life <= 0) return HLB_OK;
  compute_sponge(h);
  return h->device_ready ? upload_sponge(h) : HLB_OK;
}

}  // namespace
}  // namespace hlb

extern "C" int hlb_set_params(hlb_handle h, const hlb_params* params) {
  if (!h || !params) return fail(HLB_EINVAL, "hlb_set_params: null argument");
  if (h->device_ready) {
    // captured FP64 steps hold tau and the relaxation rates as launch arguments
    HLB_CHECK(hipStreamSynchronize(h->stream));
    h->drop_graphs();
  }
  const int rc = configure_params(h, *params, "hlb_set_params");
  return rc == HLB_OK ? refresh_sponge(h) : rc;
}

extern "C" int hlb_set_sponge(hlb_handle h, double viscosity_ratio, double width, int64_t lifetime) {
  if (!h) return fail(HLB_EINVAL, "hlb_set_sponge: null handle");
  if (h->params.kernel != HLB_KERNEL_LES)
    return fail(HLB_EINVAL, "hlb_set_sponge: the sponge layer belongs to the LES kernel (LBGKLESSpongeLayer)");
  if (!std::isfinite(viscosity_ratio) || !std::isfinite(width) || width <= 0.0)
    return fail(HLB_EINVAL, "hlb_set_sponge: the viscosity ratio must be finite and the width positive");
  if (lifetime < 0) return fail(HLB_EINVAL, "hlb_set_sponge: negative lifetime");
  if (h->device_ready) {
    // captured FP64 steps hold the sponge's arrays as launch arguments
    HLB_CHECK(hipStreamSynchronize(h->stream));
    h->drop_graphs();
  }
  h->sponge_ratio = viscosity_ratio;
  h->sponge_width = width;
  h->sponge_life = lifetime;
  if (lifetime == 0) {
    h->h_vtau.clear();  // lifetime 0: the Smagorinsky time every step
    return HLB_OK;
  }
  try {
    return refresh_sponge(h);
  } catch (const std::bad_alloc&) {
    return fail(HLB_EINVAL, "hlb_set_sponge: out of host memory");
  }
}

extern "C" int hlb_set_graphs(hlb_handle h, int enable) {
  if (!h) return fail(HLB_EINVAL, "hlb_set_graphs: null handle");
  if (h->device_ready) {
    HLB_CHECK(hipStreamSynchronize(h->stream));
    h->drop_graphs();
  }
  h->use_graph = enable != 0;
  return HLB_OK;
}

extern "C" int hlb_captured_graphs(hlb_handle h) { return h ? (int)h->graphs.size() : -1; }

extern "C" int hlb_set_iolets(hlb_handle h, const hlb_iolet_desc* inlets, int n_inlets, const hlb_iolet_desc* outlets,
                              int n_outlets) {
  if (!h) return fail(HLB_EINVAL, "hlb_set_iolets: null handle");
  try {
    const int rc = configure_iolets(h, inlets, n_inlets, outlets, n_outlets, "hlb_set_iolets");
    return rc == HLB_OK ? refresh_sponge(h) : rc;
  } catch (const std::bad_alloc&) {
    return fail(HLB_EINVAL, "hlb_set_iolets: out of host memory");
  }
}

extern "C" int hlb_get_params(hlb_handle h, hlb_params* out) {
  if (!h || !out) return fail(HLB_EINVAL, "hlb_get_params: null argument");
  *out = h->params;
  return HLB_OK;
}

extern "C" void hlb_destroy(hlb_handle h) {
  if (h && h->batch) batch_forget(h->batch, h);
  delete h;
}

extern "C" int hlb_init_equilibrium(hlb_handle h, double rho0, int64_t t0) {
  if (!h) return fail(HLB_EINVAL, "hlb_init_equilibrium: null handle");
  if (t0 < 1) return fail(HLB_EINVAL, "hlb_init_equilibrium: t0 must be >= 1");
  {
    const int rc = ensure_device(h);
    if (rc != HLB_OK) return rc;
  }
  double feq[Q];
  const FeqPre p = feq_pre(rho0, 0.0, 0.0, 0.0);
  feq_all(p, 0.0, 0.0, 0.0, feq);
  if (h->fp32()) {
    float g[Q];
    for (int j = 0; j < Q; ++j) g[j] = (float)(feq[j] - Wt(j));
    if (!h->F32.p) HLB_CHECK(h->F32.alloc((size_t)Q * h->S));
    HLB_CHECK(hipMemcpyAsync(h->feq32.p, g, sizeof g, hipMemcpyHostToDevice, h->stream));
    HLB_CHECK(launch_fill_fp32(h->F32.p, h->S, h->S, h->feq32.p, h->stream));
    HLB_CHECK(hipStreamSynchronize(h->stream));
    h->have_post = false;
    h->f_valid = true;
    h->t = t0;
    return HLB_OK;
  }
  if (!h->F.p) HLB_CHECK(h->F.alloc((size_t)Q * h->S));
  HLB_CHECK(hipMemcpyAsync(h->feq_vals.p, feq, sizeof feq, hipMemcpyHostToDevice, h->stream));
  HLB_CHECK(launch_fill_fp64(h->F.p, h->S, h->S, h->feq_vals.p, h->stream));
  HLB_CHECK(hipStreamSynchronize(h->stream));
  h->have_post = false;
  h->f_valid = true;
  h->t = t0;
  return HLB_OK;
}

extern "C" int hlb_upload_f(hlb_handle h, const double* f, int64_t t0) {
  if (!h || (!f && h->L.N > 0)) return fail(HLB_EINVAL, "hlb_upload_f: null argument");
  if (t0 < 1) return fail(HLB_EINVAL, "hlb_upload_f: t0 must be >= 1");
  {
    const int rc = ensure_device(h);
    if (rc != HLB_OK) return rc;
  }
  // The copy below replaces F: queued steps that still read it (hlb_step is
  // asynchronous, on the handle's or its batch's stream) finish first.
  if (h->batch) HLB_CHECK(hipStreamSynchronize(batch_stream(h->batch)));
  HLB_CHECK(hipStreamSynchronize(h->stream));
  const size_t count = (size_t)Q * h->S;
  if (h->fp32()) {
    if (!h->F32.p) HLB_CHECK(h->F32.alloc(count));
  } else if (!h->F.p) {
    HLB_CHECK(h->F.alloc(count));
  }
  {
    const int rc = import_sites(h, f, h->fp32() ? (void*)h->F32.p : (void*)h->F.p, h->fp32());
    if (rc != HLB_OK) return rc;
  }
  h->have_post = false;
  h->f_valid = true;
  h->t = t0;
  return HLB_OK;
}

extern "C" int hlb_step(hlb_handle h, int64_t nsteps, uint32_t flags) {
  if (!h) return fail(HLB_EINVAL, "hlb_step: null handle");
  return run_steps(h, nsteps, flags);
}

namespace hlb {
namespace {

// nsteps timed steps, replayed from a graph or launched one by one.
int timed_steps(hlb_lattice* h, int64_t nsteps, uint32_t flags, bool graph, double* ms) {
  if (!h->f_valid) return fail(HLB_EINVAL, "hlb_step_timed: no initial condition");
  HLB_CHECK(hipStreamSynchronize(h->stream));
  const bool props = (flags & HLB_STEP_PROPERTIES) != 0;
  int rc = stage_sequence(h, nsteps, props);
  if (rc != HLB_OK) return rc;
  if (graph) {
    // Capture outside the timed region: a sequence not seen before is
    // recorded by a first call that runs nothing, then replayed below.
    rc = prepare_graph(h, nsteps, props);
    if (rc != HLB_OK) return rc;
  }
  HLB_CHECK(hipEventRecord(h->ev0, h->stream));
  rc = graph ? replay_graph(h, nsteps, props) : enqueue_steps(h, nsteps, props);
  if (rc != HLB_OK) return rc;
  HLB_CHECK(hipEventRecord(h->ev1, h->stream));
  HLB_CHECK(hipEventSynchronize(h->ev1));
  float elapsed = 0.0f;
  HLB_CHECK(hipEventElapsedTime(&elapsed, h->ev0, h->ev1));
  *ms = elapsed;
  return HLB_OK;
}

}  // namespace
}  // namespace hlb

extern "C" int hlb_step_timed(hlb_handle h, int64_t nsteps, uint32_t flags, double* ms) {
  if (!h || !ms) return fail(HLB_EINVAL, "hlb_step_timed: null argument");
  if (nsteps < 0 || nsteps > kChunk) return fail(HLB_EINVAL, "hlb_step_timed: 0 to 1024 steps per timed call");
  return timed_steps(h, nsteps, flags, h->use_graph && nsteps > 0 && h->replays(nsteps), ms);
}

extern "C" int hlb_set_variant(hlb_handle h, int variant) {
  if (!h) return fail(HLB_EINVAL, "hlb_set_variant: null handle");
  const int nvar = h->fp32() ? kFp32Variants : kFp64Variants;
  if (variant < 0 || variant >= nvar) return fail(HLB_EINVAL, "hlb_set_variant: no such variant");
  if (h->device_ready) HLB_CHECK(hipStreamSynchronize(h->stream));
  h->variant = variant;
  h->variant_chosen = true;
  return HLB_OK;
}

extern "C" int hlb_variant(hlb_handle h) { return h ? h->variant : -1; }

extern "C" int hlb_autotune(hlb_handle h, int64_t trial_steps, int* variant, double* ms_per_step) {
  if (!h) return fail(HLB_EINVAL, "hlb_autotune: null handle");
  if (trial_steps < 1 || trial_steps > kChunk) return fail(HLB_EINVAL, "hlb_autotune: 1 to 1024 trial steps");
  const int before = h->variant;
  const bool chosen = h->variant_chosen;
  int best = before;
  h->variant_chosen = true;
  double best_ms = 1e300;
  const int nvar = h->fp32() ? kFp32Variants : kFp64Variants;
  // trials too short to be replayed by themselves still time what a solve's
  // sequences run
  const bool graph = h->use_graph && h->replays(std::max(trial_steps, kReplaySteps));
  for (int v = 0; v < nvar; ++v) {
    h->variant = v;
    double ms = 0.0;
    int rc = timed_steps(h, trial_steps, 0, graph, &ms);  // the first launch of a shape warms it
    if (rc == HLB_OK) rc = timed_steps(h, trial_steps, 0, graph, &ms);
    if (rc != HLB_OK) {
      h->variant = before;
      h->variant_chosen = chosen;
      return rc;
    }
    if (ms < best_ms) {
      best_ms = ms;
      best = v;
    }
  }
  h->variant = best;
  if (variant) *variant = best;
  if (ms_per_step) *ms_per_step = best_ms / (double)trial_steps;
  return HLB_OK;
}

extern "C" int hlb_synchronize(hlb_handle h) {
  if (!h) return fail(HLB_EINVAL, "hlb_synchronize: null handle");
  if (!h->device_ready) return HLB_OK;
  HLB_CHECK(hipStreamSynchronize(h->stream));
  return HLB_OK;
}

extern "C" int hlb_download_f(hlb_handle h, double* f) {
  if (!h || (!f && h->L.N > 0)) return fail(HLB_EINVAL, "hlb_download_f: null argument");
  if (!h->f_valid) return fail(HLB_EINVAL, "hlb_download_f: no state");
  const int rc = materialise_f(h);
  if (rc != HLB_OK) return rc;
  const TransferPart part{h->fp32() ? (const void*)h->F32.p : (const void*)h->F.p, Q, f};
  return export_sites(h, &part, 1, h->fp32());
}

extern "C" int hlb_get_fields(hlb_handle h, double* rho, double* u, double* wss) {
  if (!h) return fail(HLB_EINVAL, "hlb_get_fields: null handle");
  if (!h->device_ready) return fail(HLB_EINVAL, "hlb_get_fields: no state");
  const TransferPart parts[] = {{h->rho.p, 1, rho}, {h->u.p, 3, u}, {h->wss.p, 1, wss}};
  return export_sites(h, parts, 3, false);
}

namespace hlb {
namespace {

// The 17 stress planes of the state entering the next step, queued on the
// handle's stream.
int compute_stress(hlb_lattice* h, const char* who) {
  if (!h->f_valid) return fail(HLB_EINVAL, std::string(who) + ": no state");
  int rc = materialise_f(h);
  if (rc != HLB_OK) return rc;
  if (!h->stress.p) HLB_CHECK(h->stress.alloc((size_t)17 * h->S));
  const StepArgs a = make_args(h, nullptr, nullptr);
  if (h->sponge_life > 0) {
    // the relaxation time of the step the materialised state enters
    HLB_CHECK(hipStreamSynchronize(h->stream));
    const int rc = stage_iolet_values(h, h->t, 1, h->stream);
    if (rc != HLB_OK) return rc;
  }
  if (h->fp32()) HLB_CHECK(launch_stress_fp64(a, h->params.kernel, h->F32.p, true, h->stress.p, h->stream));
  else HLB_CHECK(launch_stress_fp64(a, h->params.kernel, h->F.p, false, h->stress.p, h->stream));
  return HLB_OK;
}

}  // namespace
}  // namespace hlb

extern "C" int hlb_get_stress(hlb_handle h, double* tensor, double* von_mises, double* shear_rate,
                              double* traction, double* tangential, double* normal) {
  if (!h) return fail(HLB_EINVAL, "hlb_get_stress: null handle");
  const int rc = compute_stress(h, "hlb_get_stress");
  if (rc != HLB_OK) return rc;
  const int64_t S = h->S;
  // planes: tensor 0-5, von Mises 6, shear rate 7, traction 8-10, its tangential 11-13 and normal 14-16 projections
  const double* p = h->stress.p;
  const TransferPart parts[] = {{p, 6, tensor},         {p + 6 * S, 1, von_mises},   {p + 7 * S, 1, shear_rate},
                                {p + 8 * S, 3, traction}, {p + 11 * S, 3, tangential}, {p + 14 * S, 3, normal}};
  return export_sites(h, parts, 6, false);
}

extern "C" int hlb_get_stress_rows(hlb_handle h, double* rows) {
  if (!h || (!rows && h->L.N > 0)) return fail(HLB_EINVAL, "hlb_get_stress_rows: null argument");
  const int rc = compute_stress(h, "hlb_get_stress_rows");
  if (rc != HLB_OK) return rc;
  const TransferPart part{h->stress.p, 17, rows};
  return export_sites(h, &part, 1, false);
}

extern "C" int64_t hlb_timestep(hlb_handle h) { return h ? h->t : -1; }

extern "C" int hlb_stability(hlb_handle h, int* stable) {
  if (!h || !stable) return fail(HLB_EINVAL, "hlb_stability: null argument");
  if (!h->f_valid) return fail(HLB_EINVAL, "hlb_stability: no state");
  int rc = materialise_f(h);
  if (rc != HLB_OK) return rc;
  // the scan writes its verdict straight into pinned host memory; earlier
  // work on the stream (materialise_f's) has not touched it
  volatile int* flag = reinterpret_cast<volatile int*>(h->result());
  *flag = 0;
  int* f = reinterpret_cast<int*>(h->result());
  if (h->fp32()) HLB_CHECK(launch_unstable_fp32(h->tables(), h->F32.p, h->S, f, h->stream));
  else HLB_CHECK(launch_unstable_fp64(h->tables(), h->F.p, h->S, f, h->stream));
  HLB_CHECK(hipStreamSynchronize(h->stream));
  *stable = *flag ? 0 : 1;
  return HLB_OK;
}

// How long a monitor polls for its result before it waits for the stream.  The
// wait ends ~4 us after the kernel has, and the step after it would wait for
// the staging once more (staging_idle).  One step and a monitor on a 14k-site
// pipe, with the iolet values read in place: FP64 28.5 -> 21.4 us, FP32 (which
// copies its member record) 27.2 -> 22.6; a monitor alone 17.2 -> 12.8.  Both
// passes in one launch, folded by the workgroup that ends last, took 0.8 us
// more.
constexpr std::chrono::microseconds kMonitorPoll(200);

extern "C" int hlb_monitor(hlb_handle h, double out[4]) {
  if (!h || !out) return fail(HLB_EINVAL, "hlb_monitor: null argument");
  if (!h->device_ready) return fail(HLB_EINVAL, "hlb_monitor: no state");
  if (!h->mon_scratch.p) {
    HLB_CHECK(h->mon_scratch.alloc(monitor_scratch(h->nslab)));
  }
  // the last pass writes the four results, then the word that says so, straight
  // into pinned host memory
  volatile double* arrived = h->result() + 4;
  *arrived = h->nslab > 0 ? 0.0 : 1.0;
  HLB_CHECK(launch_monitor(h->tables(), h->rho.p, h->u.p, h->S, h->mon_scratch.p, h->result(), true, h->stream));
  const auto start = std::chrono::steady_clock::now();
  while (*arrived == 0.0 && std::chrono::steady_clock::now() - start < kMonitorPoll) {
  }
  if (*arrived == 0.0) HLB_CHECK(hipStreamSynchronize(h->stream));
  std::atomic_thread_fence(std::memory_order_acquire);
  h->staging_idle = true;  // whatever was queued ahead of the monitor has run
  std::memcpy(out, h->result(), 4 * sizeof(double));
  return HLB_OK;
}

extern "C" int64_t hlb_site_count(hlb_handle h) { return h ? h->L.N : -1; }

extern "C" int hlb_class_counts(hlb_handle h, int64_t out[6]) {
  if (!h || !out) return fail(HLB_EINVAL, "hlb_class_counts: null argument");
  for (int c = 0; c < 6; ++c) out[c] = h->L.off[c + 1] - h->L.off[c];
  return HLB_OK;
}

extern "C" int hlb_site_coords(hlb_handle h, int64_t* out) {
  if (!h || !out) return fail(HLB_EINVAL, "hlb_site_coords: null argument");
  for (size_t i = 0; i < h->L.coords.size(); ++i) out[i] = h->L.coords[i];
  return HLB_OK;
}

extern "C" int hlb_neighbour_tables(hlb_handle h, int64_t* push, uint32_t* pull) {
  if (!h) return fail(HLB_EINVAL, "hlb_neighbour_tables: null handle");
  if (push) push_table(h->L, push);
  if (pull && !h->device_ready) {
    pull_table(h->L, pull);
  } else if (pull) {
    // The slots the device kernels gather from, computed by the same code
    // on the device, expressed in the reference's order (a padding slot reads as
    // 0xffffffff).
    const int64_t N = h->L.N, S = h->S;
    DevBuf<uint32_t> dev;
    HLB_CHECK(dev.alloc((size_t)18 * S));
    HLB_CHECK(launch_upstream_table(h->tables(), dev.p, S, h->stream));
    std::vector<uint32_t> tmp((size_t)18 * S);
    HLB_CHECK(hipMemcpyAsync(tmp.data(), dev.p, sizeof(uint32_t) * tmp.size(), hipMemcpyDeviceToHost, h->stream));
    HLB_CHECK(hipStreamSynchronize(h->stream));
    for (int j = 0; j < 18; ++j)
      for (int64_t k = 0; k < N; ++k) {
        uint32_t v = tmp[(size_t)j * S + h->inv[k]];
        // the boundary delegates replace what a link between fluid sites gathered
        if (h->inner_links() && ((h->L.inner[(size_t)k] >> (INV[j + 1] - 1)) & 1u)) v = (uint32_t)h->inv[k];
        pull[(size_t)j * N + k] = v < (uint32_t)S ? (uint32_t)h->perm[v] : 0xffffffffu;
      }
  }
  return HLB_OK;
}

extern "C" int hlb_site_masks(hlb_handle h, uint32_t* wall, uint32_t* iolet, int32_t* iolet_id,
                              int32_t* site_type) {
  if (!h) return fail(HLB_EINVAL, "hlb_site_masks: null handle");
  const int64_t N = h->L.N;
  for (int64_t k = 0; k < N; ++k) {
    if (wall) wall[k] = h->L.wall[k];
    if (iolet) iolet[k] = h->L.iolet[k];
    if (iolet_id) iolet_id[k] = h->L.ioletId[k];
    if (site_type) site_type[k] = h->L.siteType[k];
  }
  return HLB_OK;
}

extern "C" int hlb_wall_geometry(hlb_handle h, double* dist, double* normal) {
  if (!h) return fail(HLB_EINVAL, "hlb_wall_geometry: null handle");
  if (dist)
    for (size_t i = 0; i < h->L.q.size(); ++i) dist[i] = (double)h->L.q[i];
  if (normal)
    for (size_t i = 0; i < h->L.nrm.size(); ++i) normal[i] = (double)h->L.nrm[i];
  return HLB_OK;
}

namespace hlb {

int64_t device_bytes(const hlb_lattice* h) {
  const int64_t S = h->S, SB = h->SB, SI = h->SI;
  const int64_t fsz = h->fp32() ? 4 : 8;
  int64_t b = 3 * Q * fsz * S + Q * fsz * SI;        // A[2], F, G
  b += (int64_t)sizeof(SlabRec) * std::max<int64_t>(h->nslab, 1);  // slab records
  b += (16 + 18 * 4 + 3 * 4 + (h->inner_links() ? 4 : 0)) * SB;  // boundary records, q, normals, marked links
  b += 36 * 8 * SI + 4 * SI + 16 * h->wk_stride();    // Ladd factors, Windkessel places and two sets of terms
  b += 5 * 8 * S + 4 * h->L.N;                        // rho, u, wss, the site -> slot index
  b += 8 * h->stage_doubles();                        // member record and per-step rows
  b += (12 + 24 + 4 + (int64_t)(sizeof(WkIolet) + sizeof(WkRef))) * h->iolet_count();  // per-iolet constants and state
  b += 32 * 256;                                      // alignment of the small arrays in their allocation
  return b;
}

}  // namespace hlb

extern "C" int64_t hlb_device_bytes(hlb_handle h) { return h ? hlb::device_bytes(h) : -1; }

extern "C" int hlb_iolet_state(hlb_handle h, int outlet, int index, double out[4]) {
  if (!h || !out) return fail(HLB_EINVAL, "hlb_iolet_state: null argument");
  const int n = outlet ? h->n_out : h->n_in;
  if (index < 0 || index >= n) return fail(HLB_EINVAL, "hlb_iolet_state: no such iolet");
  const int g = outlet ? h->n_in + index : index;
  const HostIolet& io = h->iolets[g];
  if (io.IsWK() && h->device_ready) {
    WkIolet w;
    HLB_CHECK(copy_now(&w, h->wk.p + g, sizeof(WkIolet), hipMemcpyDeviceToHost, h->stream));
    out[0] = w.density;
    out[1] = w.densityNew;
    out[2] = w.flowRate;
    out[3] = w.flowRateOld;
    return HLB_OK;
  }
  std::vector<double> dens(h->iolets.size()), vmax(h->iolets.size()), vmax2(h->iolets.size());
  const int rc = iolet_values(h, std::max<int64_t>(1, h->t - 1), dens.data(), vmax.data(), vmax2.data());
  if (rc != HLB_OK) return rc;
  out[0] = io.IsWK() ? 1.0 : dens[g];
  out[1] = out[0];
  out[2] = out[3] = 0.0;
  return HLB_OK;
}

// ---- hlb_monitor_noalloc: the monitors without any device allocation ------
//
// Callers that cannot allocate device memory (code under graph capture,
// serving loops, harnesses that forbid hipMalloc) get the monitors from a
// fixed scratch array in the library's own device memory: the per-workgroup
// partials from offset 0, the four results in the last 256 bytes.  Every
// handle on a GPU shares that GPU's array, so calls that overlap on one GPU
// race; each call fully writes what it reads back, so nothing needs clearing.

constexpr size_t kScratchBytes = size_t(16) << 20;  // 16 MiB per GPU
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace hlb {
namespace {

constexpr size_t kScratchOut = kScratchBytes - 256;  // the four results

std::mutex g_scratch_mu;
std::vector<unsigned char*> g_scratch_ptr;  // per device, resolved once

// The device address of `scratch` on `device`, which must be current.
int scratch_ptr(int device, unsigned char** out) {
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (device < 0) return fail(HLB_EINVAL, "hlb_monitor_noalloc: no device");
  if ((size_t)device >= g_scratch_ptr.size()) g_scratch_ptr.resize((size_t)device + 1, nullptr);
  if (!g_scratch_ptr[(size_t)device]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return dev_fail(e != hipSuccess ? e : hipErrorInvalidSymbol, "hipGetSymbolAddress(scratch)");
    g_scratch_ptr[(size_t)device] = static_cast<unsigned char*>(p);
  }
  *out = g_scratch_ptr[(size_t)device];
  return HLB_OK;
}

}  // namespace
}  // namespace hlb

extern "C" int64_t hlb_noalloc_scratch_bytes(void) { return (int64_t)kScratchBytes; }

extern "C" int hlb_monitor_noalloc(hlb_handle h, double out[4]) {
  if (!h || !out) return fail(HLB_EINVAL, "hlb_monitor_noalloc: null argument");
  if (!h->device_ready) return fail(HLB_EINVAL, "hlb_monitor_noalloc: no state");
  const size_t need = monitor_scratch(h->nslab);
  if (need > kScratchOut)
    return fail(HLB_ERANGE, "hlb_monitor_noalloc: the lattice needs " + std::to_string(need) +
                                " bytes of partials, more than the " + std::to_string(kScratchOut) +
                                " the fixed scratch holds (" + std::to_string(h->nslab) + " slabs); use hlb_monitor");
  int cur = -1;
  HLB_CHECK(hipGetDevice(&cur));
  if (cur != h->device) HLB_CHECK(hipSetDevice(h->device));
  unsigned char* base = nullptr;
  int rc = scratch_ptr(h->device, &base);
  if (rc == HLB_OK) {
    double* dout = reinterpret_cast<double*>(base + kScratchOut);
    hipError_t e = launch_monitor(h->tables(), h->rho.p, h->u.p, h->S, base, dout, false, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(out, dout, 4 * sizeof(double), hipMemcpyDeviceToHost, h->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
    if (e != hipSuccess) rc = dev_fail(e, "hlb_monitor_noalloc");
  }
  if (cur != h->device) (void)hipSetDevice(cur);
  return rc;
}
