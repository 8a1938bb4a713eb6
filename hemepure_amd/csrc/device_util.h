// device_util.h -- addressing helpers shared by the step kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "d3q19.h"
#include "lbm_kernels.h"

namespace hlb {

constexpr int kBlock = 256;  // threads (device slots) per workgroup tile

// Loads and stores through a uniform plane base and a 32-bit element index:
// the byte offset stays 32-bit (planes are < 2^29 elements, checked at
// create time), so the address is an SGPR base plus one VGPR offset.  The
// casts name the global address space: pointers read from a table in memory
// would otherwise be generic and compile to flat accesses.
#define HLB_GLOBAL __attribute__((address_space(1)))

template <typename T>
__device__ __forceinline__ T ldp(const T* base, uint32_t i) {
  const char* p = reinterpret_cast<const char*>(base) + i * (uint32_t)sizeof(T);
  return *(const HLB_GLOBAL T*)p;
}
template <typename T>
__device__ __forceinline__ T ldp_nt(const T* base, uint32_t i) {
  const char* p = reinterpret_cast<const char*>(base) + i * (uint32_t)sizeof(T);
  return __builtin_nontemporal_load((const HLB_GLOBAL T*)p);
}
template <typename T>
__device__ __forceinline__ void stp_nt(T* base, uint32_t i, T v) {
  char* p = reinterpret_cast<char*>(base) + i * (uint32_t)sizeof(T);
  __builtin_nontemporal_store(v, (HLB_GLOBAL T*)p);
}
template <typename T>
__device__ __forceinline__ void stp(T* base, uint32_t i, T v) {
  char* p = reinterpret_cast<char*>(base) + i * (uint32_t)sizeof(T);
  *(HLB_GLOBAL T*)p = v;
}

template <typename T>
__device__ __forceinline__ T* plane(T* p, int64_t S, int j) {
  return p + (int64_t)j * S;
}

// Tile orders over the workgroups behind the first `lead` ones (a multiple of
// the XCD count, so a workgroup's XCD stays its index mod 8).
// XCD-contiguous: the hardware hands workgroup w to XCD w mod 8, so logical
// tile (w mod 8) * (grid / 8) + w / 8 gives each XCD one contiguous eighth of
// the tiles (grid is a multiple of 8).
__device__ __forceinline__ uint32_t xcd_tile(uint32_t lead = 0) {
  const uint32_t w = blockIdx.x - lead, per = (gridDim.x - lead) / kXcds;
  return (w % kXcds) * per + w / kXcds;
}

// XCD chunks: XCD x's k-th workgroup takes tile k mod C of chunk x + 8 (k / C),
// C = kXcdChunk, so chunks of C consecutive tiles go to the XCDs in turn (grid
// is a multiple of 8 C; a bijection on [0, grid)).
__device__ __forceinline__ uint32_t xcd_chunk_tile(uint32_t lead = 0) {
  const uint32_t w = blockIdx.x - lead, x = w % kXcds, k = w / kXcds;
  return (x + kXcds * (k / kXcdChunk)) * kXcdChunk + k % kXcdChunk;
}

// The logical tile of this workgroup in tile order ORDER (a TileOrder).
template <int ORDER>
__device__ __forceinline__ uint32_t tile_index(uint32_t lead) {
  if constexpr (ORDER == kOrderXcd) return xcd_tile(lead);
  else if constexpr (ORDER == kOrderXcdChunks) return xcd_chunk_tile(lead);
  else return blockIdx.x - lead;
}

__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}

// Plane j of a wave-uniform array, made an opaque scalar value so every
// access is (scalar base) + (32-bit lane offset) rather than a 64-bit vector
// address the compiler rebuilds per plane.
template <typename T>
__device__ __forceinline__ T* uplane(T* p, int64_t S, int j) {
  return reinterpret_cast<T*>(uniform64(reinterpret_cast<uint64_t>(p + (int64_t)j * S)));
}

// One lane of a slab: its slot, block-local (y, z) and boundary index.
struct Lane {
  uint32_t r;              // slab record (wave-uniform)
  uint32_t slot;
  int y, z;
  bool boundary;
  uint32_t b;              // compact boundary index (valid when boundary)
  uint64_t fm[kReach];     // reachable slabs' fluid masks (wave-uniform)
  int32_t base[kReach];    // and their first slots
};

// Number of set bits of the wave-uniform mask below this lane, plus add.
__device__ __forceinline__ uint32_t mbcnt64(uint64_t mask, uint32_t add) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, add));
}

// Decodes slab record r for this lane; false for a position that is not
// fluid or a record past the end (the lane has nothing to do).  r must be
// wave-uniform; the record is read with scalar loads that do not wait on one
// another.
__device__ __forceinline__ bool slab_lane(const BrickTables& bt, uint32_t r, Lane& L) {
  if (r >= (uint64_t)bt.nslab) return false;
  const uint32_t lane = threadIdx.x & 63u;
  const HLB_GLOBAL SlabRec* g = (const HLB_GLOBAL SlabRec*)(bt.rec + r);
#pragma unroll
  for (int k = 0; k < kReach; ++k) {
    L.fm[k] = uniform64(g->fm[k]);
    L.base[k] = __builtin_amdgcn_readfirstlane(g->base[k]);
  }
  const uint64_t bm = uniform64(g->bmask);
  const int32_t bbase = __builtin_amdgcn_readfirstlane(g->bbase);
  const uint64_t fm = L.fm[reach_entry(0, 0, 0)];
  if (!((fm >> lane) & 1u)) return false;
  L.r = r;
  L.y = (int)(lane >> 3);
  L.z = (int)(lane & 7u);
  L.slot = mbcnt64(fm, (uint32_t)L.base[reach_entry(0, 0, 0)]);
  L.boundary = (bm >> lane) & 1u;
  L.b = L.boundary ? mbcnt64(bm, (uint32_t)bbase) : 0u;
  return true;
}

// Index among the lanes of the slab set in mask (uniform) below this lane.
__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  const uint32_t lane = threadIdx.x & 63u;
  return (uint32_t)__builtin_popcountll(mask & ((1ull << lane) - 1ull));
}

// Slot of position lane + DELTA of a slab with fluid mask m and first slot
// base; fluid receives m shifted so that bit `lane` says whether that
// position is fluid.  m and base are wave-uniform, so the shift and the count
// of fluid positions below DELTA are scalar work and the per-lane count is
// one mbcnt pair.
template <int DELTA>
__device__ __forceinline__ uint32_t shifted_slot(uint64_t m, uint32_t base, uint64_t& fluid) {
  uint64_t ms = m;
  uint32_t add = base;
  if constexpr (DELTA > 0) {
    ms = m >> DELTA;
    add += (uint32_t)__builtin_popcountll(m & ((1ull << DELTA) - 1ull));
  } else if constexpr (DELTA < 0) {
    ms = m << (-DELTA);
  }
  fluid = ms;
  return mbcnt64(ms, add);
}

// Lanes at a brick face: y = 0, y = 7, z = 0, z = 7 (lane = y * 8 + z).
constexpr uint64_t kLanesY0 = 0x00000000000000ffull, kLanesY7 = 0xff00000000000000ull;
constexpr uint64_t kLanesZ0 = 0x0101010101010101ull, kLanesZ7 = 0x8080808080808080ull;

// Slot of the upstream site x - c_J of a lane (pull direction J) where that
// position is fluid; fluid_lanes receives the lane mask of the lanes for
// which it is (for the others the link is a wall or iolet link and the slot
// is meaningless; upstream_slot substitutes the lane's own).  The position is
// lane + 8 oy + oz in the slab the record names for the x step, or -- for
// lanes whose y / z step leaves the brick -- 64 or 8 positions back in the
// neighbouring brick's slab: at most four candidates, each one mbcnt pair,
// picked with constant lane masks; the fluid test combines the candidates'
// shifted masks with scalar logic into one lane mask.  plus (wave-uniform) is
// added to every candidate's base, scalar work as well.
template <int J>
__device__ __forceinline__ uint32_t upstream_pos(const Lane& L, uint64_t& fluid_lanes, uint32_t plus = 0) {
  constexpr int ox = -CX[J], oy = -CY[J], oz = -CZ[J];
  constexpr int d00 = 8 * oy + oz;
  // lanes whose step leaves the brick in y / in z
  constexpr uint64_t Y = oy == 0 ? 0ull : (oy < 0 ? kLanesY0 : kLanesY7);
  constexpr uint64_t Z = oz == 0 ? 0ull : (oz < 0 ? kLanesZ0 : kLanesZ7);
  const bool yo = __builtin_amdgcn_inverse_ballot_w64(Y);
  const bool zo = __builtin_amdgcn_inverse_ballot_w64(Z);
  // constant entry indices only, so the masks and bases stay in scalar registers
  constexpr int e00 = reach_entry(ox, 0, 0);
  uint64_t m00 = 0;
  uint32_t slot = shifted_slot<d00>(L.fm[e00], (uint32_t)L.base[e00] + plus, m00);
  uint64_t fluid = m00 & ~(Y | Z);
  if constexpr (oy != 0 && oz != 0) {
    static_assert(ox == 0, "D3Q19 links have at most two nonzero components");
    constexpr int e10 = reach_entry(0, oy, 0), e01 = reach_entry(0, 0, oz), e11 = reach_entry(0, oy, oz);
    uint64_t m10 = 0, m01 = 0, m11 = 0;
    const uint32_t s10 = shifted_slot<d00 - 64 * oy>(L.fm[e10], (uint32_t)L.base[e10] + plus, m10);
    const uint32_t s01 = shifted_slot<d00 - 8 * oz>(L.fm[e01], (uint32_t)L.base[e01] + plus, m01);
    const uint32_t s11 = shifted_slot<d00 - 64 * oy - 8 * oz>(L.fm[e11], (uint32_t)L.base[e11] + plus, m11);
    slot = yo ? (zo ? s11 : s10) : (zo ? s01 : slot);
    fluid |= (m10 & (Y & ~Z)) | (m01 & (Z & ~Y)) | (m11 & (Y & Z));
  } else if constexpr (oy != 0) {
    constexpr int e10 = reach_entry(ox, oy, 0);
    uint64_t m10 = 0;
    const uint32_t s10 = shifted_slot<d00 - 64 * oy>(L.fm[e10], (uint32_t)L.base[e10] + plus, m10);
    slot = yo ? s10 : slot;
    fluid |= m10 & Y;
  } else if constexpr (oz != 0) {
    constexpr int e01 = reach_entry(ox, 0, oz);
    uint64_t m01 = 0;
    const uint32_t s01 = shifted_slot<d00 - 8 * oz>(L.fm[e01], (uint32_t)L.base[e01] + plus, m01);
    slot = zo ? s01 : slot;
    fluid |= m01 & Z;
  }
  fluid_lanes = fluid;
  return slot;
}

// The steady step's gather of pull direction J.  The planes of an opposite
// pair (J, INV[J]) are adjacent, so both are reached from the lower one with a
// 32-bit element offset (2 S elements; see launch_step_fp64 for FP64's limit):
// where the upstream position is not fluid (a wall or iolet link ib = INV[J])
// the lane reads its own value in plane ib -- the bounce-back value, which SBB
// keeps, BFL keeps or interpolates from and iolet and GZS links replace -- so
// no boundary delegate loads it, except for a link between two fluid sites
// (kInnerLinks), where the upstream position is fluid.  The pair's plane
// offset is folded into the scalar bases, and own[k] (the own slot in the k-th
// plane of a pair) into two values a lane forms once, so the choice costs one
// select.
template <int J, typename T>
__device__ __forceinline__ T gather_bb(const T* lower, uint32_t S, const Lane& L, const uint32_t (&own)[2]) {
  constexpr bool upper = J > INV[J];
  uint64_t fluid = 0;
  const uint32_t up = upstream_pos<J>(L, fluid, upper ? S : 0u);
  return ldp(lower, __builtin_amdgcn_inverse_ballot_w64(fluid) ? up : own[upper ? 0 : 1]);
}

// Velocity iolet links whose profile factors are loaded together: in groups of
// three the delegate needs no more registers than the collision.
constexpr int kLaddGroup = 3;

// A boundary site's record (BndRec), read with one 16-byte load.
struct Bnd {
  uint32_t far, near, iolet, gi, ii;
  bool wall;
};
__device__ __forceinline__ Bnd no_bnd() { return Bnd{0, 0, 0, 0, 0, false}; }
__device__ __forceinline__ Bnd load_bnd(const BndRec* rec, uint32_t b) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 v = *(const HLB_GLOBAL u32x4*)(rec + b);
  return Bnd{v.x & (kLinkBits | kInnerLinks), v.y & kLinkBits, v.z, v.y >> 18, v.w, (v.x >> 31) != 0};
}

// Where the value of iolet link d goes, which is what the next step gathers in
// direction INV[d]: into the site's own post-collision row, plane d.  Nothing but
// the site's own bounce-back gather (gather_bb) reads it there: no site lies
// downstream of an iolet link, or one that does has the link from its side too
// and replaces what it gathered (kInnerLinks).  So the next step has no load
// of its own for it.  BFL's interpolation with the site's own value (a wall link
// opposite the iolet link, far bit d) needs the post-collision value in that
// place; the iolet's then goes to G.
// With every value in G the waves of an iolet layer, which decide a small
// lattice's step, had one more round of loads (boundary record, iolet index, G)
// ahead of the collision: 30k-site cylinder FP64 5.98 -> 5.50 us a step, FP32
// 5.67 -> 5.06, a 45k-site bifurcation with BFL walls 8.25 -> 8.04 (FP32) and
// 9.11 -> 9.06, the 0.70M-site one 40.4 -> 40.25; larger lattices unchanged.
template <typename T>
__device__ __forceinline__ T* iolet_place(int d, T* row, uint32_t slot, T* G, int64_t SI, const Bnd& r) {
  return (r.far & (1u << (d - 1))) ? plane(G, SI, INV[d]) + r.ii : row + slot;
}

template <int J>
__device__ __forceinline__ uint32_t upstream_slot(const Lane& L) {
  uint64_t fluid = 0;
  const uint32_t slot = upstream_pos<J>(L, fluid);
  return __builtin_amdgcn_inverse_ballot_w64(fluid) ? slot : L.slot;
}

}  // namespace hlb
