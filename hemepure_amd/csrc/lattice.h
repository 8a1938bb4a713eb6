// lattice.h -- host-side LatticeData: site classification and the reference's
// class-major site order.
#pragma once

#include <cstdint>
#include <vector>

#include "../../include/hemepure_amd.h"
#include "parallel.h"

namespace hlb {

// SiteType (src/geometry/SiteType.h:17-24).
enum : int32_t { kSolidType = 0, kFluidType = 1, kInletType = 2, kOutletType = 3 };

// Cell of position (x, y, z) within its block of side bs, z fastest; the cells of
// a block of side 1291 no longer fit 32 bits.
template <typename T>
int64_t cell_in_block(T x, T y, T z, T bs) {
  return ((int64_t)(x % bs) * bs + y % bs) * bs + z % bs;
}

struct HostLattice {
  int32_t blocks[3] = {0, 0, 0};
  int32_t bs = 8;
  int64_t N = 0;
  int64_t off[7] = {0, 0, 0, 0, 0, 0, 0};  // class c occupies [off[c], off[c+1])
  RawVector<int32_t> coords;   // N*3
  RawVector<uint32_t> wall;    // N, bit d-1 set for a wall link d
  RawVector<uint32_t> iolet;   // N, bit d-1 set for an inlet/outlet link d
  RawVector<int32_t> ioletId;  // N
  RawVector<int32_t> siteType; // N
  int64_t links = 0;           // wall and iolet links, all sites
  // N, bit d-1 set for a wall or iolet link d that leads to a fluid site; empty
  // when no link does (mark_inner_links).
  RawVector<uint32_t> inner;
  RawVector<float> q;          // N*18 link distances as read
  RawVector<float> nrm;        // N*3 wall normal normalised in float (+inf if none)
  // Site map: per block a slot (or -1), per slot the block's contiguous indices (or -1).
  std::vector<int64_t> blockSlot;
  RawVector<int32_t> slotSites;

  int64_t site_at(int64_t x, int64_t y, int64_t z) const;
  int collision_class(int64_t k) const;
};

// Builds the lattice; returns HLB_OK or an HLB_E* code with hlb_last_error set.
int build_lattice(const hlb_geometry& g, HostLattice& L);

// Fills L.inner.
void mark_inner_links(HostLattice& L);

// The pull table, 18*N: source of direction j = 1..18, or the site itself.
void pull_table(const HostLattice& L, uint32_t* out);

// The reference's push table (n*19 int64, rubbish slot n*19), from the site map.
void push_table(const HostLattice& L, int64_t* out);

}  // namespace hlb
