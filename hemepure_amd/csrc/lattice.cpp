// lattice.cpp -- LatticeData construction for one GPU (one rank: every site is
// mid-domain, there are no halo slots).
//
// Classification follows SiteData::SiteData (src/geometry/SiteDataBare.cc:24-76)
// and the collision-class switch of LatticeData::ProcessReadSites
// (src/geometry/LatticeData.cc:220-240); the contiguous order is class-major,
// then block order, then site-in-block order, both z-fastest
// (LatticeData.h:375-436, src/geometry/VolumeTraverser.cc:56-70).
//
// The pull table inverts the reference's push table on plain links: for site k
// and direction j, the value arriving along j comes from the fluid site at
// x_k - c_j exactly when k's link INV[j] is a plain link.  Otherwise a
// boundary delegate of site k itself writes it (SimpleBounceBack, BFL, Nash,
// Ladd all write fNew[k*19 + INV[d]] for their link d).  Each (site, j) slot
// must have exactly one writer in the reference's push step; geometries where
// the two sides of a link disagree give zero or two writers and are rejected.  A
// link that is a wall or an iolet from both sides has one writer whether or not
// there is fluid beyond it: two sites with a wall of no thickness between them.
#include "lattice.h"

#include <atomic>
#include <cmath>
#include <limits>
#include <string>
#include <unordered_set>

#include "d3q19.h"
#include "errors.h"
#include "parallel.h"

namespace hlb {

int64_t HostLattice::site_at(int64_t x, int64_t y, int64_t z) const {
  const int64_t SX = (int64_t)blocks[0] * bs, SY = (int64_t)blocks[1] * bs, SZ = (int64_t)blocks[2] * bs;
  if (x < 0 || y < 0 || z < 0 || x >= SX || y >= SY || z >= SZ) return -1;
  const int64_t b = ((x / bs) * blocks[1] + (y / bs)) * blocks[2] + (z / bs);
  const int64_t slot = blockSlot[b];
  if (slot < 0) return -1;
  return slotSites[slot * (int64_t)bs * bs * bs + cell_in_block<int64_t>(x, y, z, bs)];
}

int HostLattice::collision_class(int64_t k) const {
  for (int c = 0; c < 6; ++c)
    if (k < off[c + 1]) return c;
  return 5;
}

namespace {

// Vector3D<float>::GetNormalised (src/util/Vector3D.h:237-265), float math.
void normalise_float(float v[3]) {
  if (v[0] == 0.0f && v[1] == 0.0f && v[2] == 0.0f) return;
  const float mag = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
  v[0] /= mag;
  v[1] /= mag;
  v[2] /= mag;
}

// The first inconsistent record, in input order, of a geometry known to hold
// one.
int site_map_error(const hlb_geometry& g) {
  const int64_t SX = (int64_t)g.blocks[0] * g.block_size, SY = (int64_t)g.blocks[1] * g.block_size,
                SZ = (int64_t)g.blocks[2] * g.block_size;
  std::unordered_set<int64_t> seen;
  for (int64_t i = 0; i < g.n_sites; ++i) {
    const int64_t x = g.coords[3 * i], y = g.coords[3 * i + 1], z = g.coords[3 * i + 2];
    if (x < 0 || y < 0 || z < 0 || x >= SX || y >= SY || z >= SZ)
      return fail(HLB_EGEOMETRY, "hlb_create: site outside the block grid");
    if (!seen.insert((x * SY + y) * SZ + z).second) return fail(HLB_EGEOMETRY, "hlb_create: duplicate fluid site");
  }
  return HLB_OK;
}

// The link type of contiguous site k in direction d (1..18).
uint8_t link_of(const HostLattice& L, int64_t k, int d) {
  if ((L.wall[k] >> (d - 1)) & 1u) return HLB_LINK_WALL;
  if ((L.iolet[k] >> (d - 1)) & 1u) return HLB_LINK_INLET;
  return HLB_LINK_NONE;
}

// The lowest site (and its lowest direction) of a lattice known to hold a
// distribution with no writer or two.
int one_writer_error(const HostLattice& L) {
  for (int64_t k = 0; k < L.N; ++k) {
    const int64_t x = L.coords[3 * k], y = L.coords[3 * k + 1], z = L.coords[3 * k + 2];
    for (int j = 1; j < Q; ++j) {
      const int ib = INV[j];
      const int64_t src = L.site_at(x - CX[j], y - CY[j], z - CZ[j]);
      const bool plain = link_of(L, k, ib) == HLB_LINK_NONE;
      const bool srcPushes = src >= 0 && link_of(L, src, j) == HLB_LINK_NONE;
      if (plain != srcPushes)
        return fail(HLB_EGEOMETRY, "hlb_create: link type disagrees with neighbour fluidity at site (" +
                                       std::to_string(x) + "," + std::to_string(y) + "," + std::to_string(z) +
                                       ") direction " + std::to_string(ib) +
                                       " (the push step would write that distribution " + (plain ? "zero" : "two") +
                                       " times)");
    }
  }
  return HLB_OK;
}

}  // namespace

int build_lattice(const hlb_geometry& g, HostLattice& L) {
  if (g.block_size <= 0 || g.blocks[0] <= 0 || g.blocks[1] <= 0 || g.blocks[2] <= 0 || g.n_sites < 0)
    return fail(HLB_EINVAL, "hlb_create: bad block grid");
  if (g.n_sites > 0 && (!g.coords || !g.link_type || !g.link_iolet || !g.link_dist || !g.normal_avail ||
                        !g.normal))
    return fail(HLB_EINVAL, "hlb_create: null geometry array");
  // Device planes are addressed with 32-bit byte offsets (8-byte elements).
  if (g.n_sites > (int64_t(1) << 29) - 64)
    return fail(HLB_EINVAL, "hlb_create: more than 2^29-64 sites per handle");
  for (int a = 0; a < 3; ++a) L.blocks[a] = g.blocks[a];
  L.bs = g.block_size;
  const int64_t bs = g.block_size, spb = bs * bs * bs;
  const int64_t BX = g.blocks[0], BY = g.blocks[1], BZ = g.blocks[2];
  const int64_t SX = BX * bs, SY = BY * bs, SZ = BZ * bs;
  const int64_t n = g.n_sites;

  // Site map over the input records: the occupied blocks, numbered in block
  // order, then each record's cell in its block.
  std::atomic<bool> bad{false};
  L.blockSlot.assign((size_t)(BX * BY * BZ), -1);
  parallel_ranges(n, [&](int, int64_t lo, int64_t hi) {
    for (int64_t i = lo; i < hi; ++i) {
      const int32_t x = g.coords[3 * i], y = g.coords[3 * i + 1], z = g.coords[3 * i + 2];
      if (x < 0 || y < 0 || z < 0 || x >= SX || y >= SY || z >= SZ) {
        bad.store(true, std::memory_order_relaxed);
        return;
      }
      int64_t& slot = L.blockSlot[(size_t)(((x / (int32_t)bs) * BY + (y / (int32_t)bs)) * BZ + (z / (int32_t)bs))];
      if (__atomic_load_n(&slot, __ATOMIC_RELAXED) != 0) __atomic_store_n(&slot, int64_t(0), __ATOMIC_RELAXED);
    }
  });
  if (bad.load()) return site_map_error(g);
  std::vector<int64_t> slotBlock;
  for (int64_t b = 0; b < BX * BY * BZ; ++b)
    if (L.blockSlot[(size_t)b] == 0) {
      L.blockSlot[(size_t)b] = (int64_t)slotBlock.size();
      slotBlock.push_back(b);
    }
  const int64_t nslot = (int64_t)slotBlock.size(), cells = nslot * spb;
  // Cells are shared out in parts of `per`: whole blocks, or the x layers of large
  // ones, of which there may be few.
  const int64_t per = spb > 4096 ? bs * bs : spb, parts = cells / per;
  // Mostly empty blocks: by sites where cells need not be looked at.  us per
  // lattice, by cells / by sites (8 cores): 729 sites in 262,144 cells 720 / 490, in
  // 32,768 200 / 253, 27,000 sites in 262,144 cells 3,270 / 7,250.
  const bool sparse = n * 32 < cells;
  const int64_t partGrain = std::max<int64_t>(1, (sparse ? 16 * kGrain : kGrain) / per);
  RawVector<int32_t> cellInput;
  cellInput.resize((size_t)cells);
  parallel_ranges(parts, [&](int, int64_t lo, int64_t hi) {
    std::fill(cellInput.begin() + lo * per, cellInput.begin() + hi * per, -1);
  }, partGrain);
  auto cell_of = [&](int64_t i) {
    const uint32_t b = (uint32_t)bs;
    const uint32_t x = g.coords[3 * i], y = g.coords[3 * i + 1], z = g.coords[3 * i + 2];  // checked: not negative
    return L.blockSlot[(size_t)(((x / b) * BY + (y / b)) * BZ + (z / b))] * spb + cell_in_block(x, y, z, b);
  };
  parallel_ranges(n, [&](int, int64_t lo, int64_t hi) {
    for (int64_t i = lo; i < hi; ++i) {
      int32_t* cell = &cellInput[(size_t)cell_of(i)];
      if (__atomic_exchange_n(cell, (int32_t)i, __ATOMIC_RELAXED) >= 0) {
        bad.store(true, std::memory_order_relaxed);
        return;
      }
    }
  });
  if (bad.load()) return site_map_error(g);

  // Classification of every input record.
  RawVector<uint32_t> wall, iol;
  RawVector<int32_t> ioletId, type;
  RawVector<uint8_t> cls;
  wall.resize((size_t)n);
  iol.resize((size_t)n);
  ioletId.resize((size_t)n);
  type.resize((size_t)n);
  cls.resize((size_t)n);
  std::atomic<int64_t> links{0};
  parallel_ranges(n, [&](int, int64_t lo, int64_t hi) {
    int64_t count = 0;
    for (int64_t i = lo; i < hi; ++i) {
      bool hadInlet = false, hadOutlet = false;
      uint32_t w = 0, io = 0;
      int32_t id = -1;
      for (int d = 1; d < Q; ++d) {
        const uint8_t t = g.link_type[i * 18 + d - 1];
        if (t == HLB_LINK_NONE) continue;
        ++count;
        if (t > HLB_LINK_OUTLET) {
          bad.store(true, std::memory_order_relaxed);
          return;
        }
        if (t == HLB_LINK_WALL) {
          w |= 1u << (d - 1);
          continue;
        }
        io |= 1u << (d - 1);
        id = g.link_iolet[i * 18 + d - 1];
        (t == HLB_LINK_INLET ? hadInlet : hadOutlet) = true;
      }
      wall[i] = w;
      iol[i] = io;
      ioletId[i] = id;
      type[i] = hadInlet ? kInletType : (hadOutlet ? kOutletType : kFluidType);
      const bool wl = w != 0;
      cls[i] = type[i] == kFluidType ? (wl ? 1 : 0) : type[i] == kInletType ? (wl ? 4 : 2) : (wl ? 5 : 3);
    }
    links.fetch_add(count, std::memory_order_relaxed);
  });
  if (bad.load()) return fail(HLB_EGEOMETRY, "hlb_create: unknown link type");
  L.links = links.load();

  // Class-major contiguous order: per part and class the first index, then
  // every cell's.  cellLinks: a cell's wall and iolet links, bit 31 where it is
  // fluid, for the check by blocks.
  constexpr uint32_t kFluid = 1u << 31;
  const bool by_block = spb > 1 && !sparse;
  std::vector<int64_t> next((size_t)parts * 6, 0);
  if (sparse)
    for (int64_t i = 0; i < n; ++i) next[(size_t)(cell_of(i) / per * 6 + cls[(size_t)i])]++;
  else
    parallel_ranges(parts, [&](int, int64_t lo, int64_t hi) {
      for (int64_t s = lo; s < hi; ++s)
        for (int64_t c = s * per; c < (s + 1) * per; ++c)
          if (cellInput[(size_t)c] >= 0) next[(size_t)(s * 6 + cls[(size_t)cellInput[(size_t)c]])]++;
    }, partGrain);
  L.N = n;
  int64_t k = 0;
  for (int c = 0; c < 6; ++c) {
    L.off[c] = k;
    for (int64_t s = 0; s < parts; ++s) {
      const int64_t count = next[(size_t)(s * 6 + c)];
      next[(size_t)(s * 6 + c)] = k;
      k += count;
    }
  }
  L.off[6] = k;
  RawVector<uint32_t> cellLinks;
  if (by_block) cellLinks.resize((size_t)cells);
  L.slotSites.resize((size_t)cells);
  L.coords.resize((size_t)n * 3);
  L.wall.resize((size_t)n);
  L.iolet.resize((size_t)n);
  L.ioletId.resize((size_t)n);
  L.siteType.resize((size_t)n);
  L.q.resize((size_t)n * 18);
  L.nrm.resize((size_t)n * 3);
  parallel_ranges(parts, [&](int, int64_t lo, int64_t hi) {
    for (int64_t s = lo; s < hi; ++s)
      for (int64_t c = s * per; c < (s + 1) * per; ++c) {
        const int64_t i = cellInput[(size_t)c];
        if (i < 0) {
          L.slotSites[(size_t)c] = -1;
          if (by_block) cellLinks[(size_t)c] = 0;
          continue;
        }
        const int64_t to = next[(size_t)(s * 6 + cls[(size_t)i])]++;
        L.slotSites[(size_t)c] = (int32_t)to;
        if (by_block) cellLinks[(size_t)c] = wall[(size_t)i] | iol[(size_t)i] | kFluid;
        for (int a = 0; a < 3; ++a) L.coords[(size_t)(3 * to + a)] = g.coords[3 * i + a];
        L.wall[(size_t)to] = wall[(size_t)i];
        L.iolet[(size_t)to] = iol[(size_t)i];
        L.ioletId[(size_t)to] = ioletId[(size_t)i];
        L.siteType[(size_t)to] = type[(size_t)i];
        for (int d = 0; d < 18; ++d) L.q[(size_t)(to * 18 + d)] = g.link_dist[i * 18 + d];
        float v[3];
        if (g.normal_avail[i]) {
          for (int a = 0; a < 3; ++a) v[a] = g.normal[3 * i + a];
          normalise_float(v);
        } else {
          v[0] = v[1] = v[2] = std::numeric_limits<float>::infinity();  // float(NO_VALUE)
        }
        for (int a = 0; a < 3; ++a) L.nrm[(size_t)(3 * to + a)] = v[a];
      }
  }, partGrain);

  // The one-writer check: a plain link's neighbour must be fluid with a plain
  // link back, any other link's must not push here.  Cell by cell with the blocks
  // around found once, unless a block is one cell (27,000 sites 7,950 / 7,280 us; of
  // two a side 3,600 / 7,030) or blocks are mostly empty.
  auto mismatch = [](uint32_t here, uint32_t src, int j) {
    const bool plain = !((here >> (INV[j] - 1)) & 1u);
    const bool srcPushes = (src & kFluid) && !((src >> (j - 1)) & 1u);
    return plain != srcPushes;
  };
  if (!by_block) {
    parallel_ranges(n, [&](int, int64_t lo, int64_t hi) {
      for (int64_t k = lo; k < hi; ++k) {
        const int64_t x = L.coords[3 * k], y = L.coords[3 * k + 1], z = L.coords[3 * k + 2];
        const uint32_t here = L.wall[(size_t)k] | L.iolet[(size_t)k];
        for (int j = 1; j < Q; ++j) {
          const int64_t s = L.site_at(x - CX[j], y - CY[j], z - CZ[j]);
          if (mismatch(here, s < 0 ? 0 : L.wall[(size_t)s] | L.iolet[(size_t)s] | kFluid, j)) {
            bad.store(true, std::memory_order_relaxed);
            return;
          }
        }
      }
    });
    return bad.load() ? one_writer_error(L) : HLB_OK;
  }
  parallel_ranges(parts, [&](int, int64_t lo, int64_t hi) {
    for (int64_t s = lo; s < hi; ++s) {
      const int64_t first = s * per % spb;  // of the block's cells
      const int64_t b = slotBlock[(size_t)(s * per / spb)], bx = b / (BY * BZ), by = (b / BZ) % BY, bz = b % BZ;
      const uint32_t* around[27];  // the 3 x 3 x 3 blocks' cells
      for (int e = 0; e < 27; ++e) {
        const int64_t x = bx + e / 9 - 1, y = by + (e / 3) % 3 - 1, z = bz + e % 3 - 1;
        const bool in = x >= 0 && y >= 0 && z >= 0 && x < BX && y < BY && z < BZ;
        const int64_t t = in ? L.blockSlot[(size_t)((x * BY + y) * BZ + z)] : -1;
        around[e] = t < 0 ? nullptr : &cellLinks[(size_t)(t * spb)];
      }
      const uint32_t* own = around[13];
      for (int64_t x = first / (bs * bs); x < (first + per) / (bs * bs); ++x)
        for (int64_t y = 0; y < bs; ++y)
          for (int64_t z = 0; z < bs; ++z) {
            const int64_t c = (x * bs + y) * bs + z;
            const uint32_t here = own[c];
            if (!(here & kFluid)) continue;
            const bool inner = x > 0 && y > 0 && z > 0 && x < bs - 1 && y < bs - 1 && z < bs - 1;
            for (int j = 1; j < Q; ++j) {
              uint32_t src = 0;
              if (inner) {
                src = own[c - ((CX[j] * bs + CY[j]) * bs + CZ[j])];
              } else {
                int64_t p[3] = {x - CX[j], y - CY[j], z - CZ[j]};
                int e = 13;
                const int step[3] = {9, 3, 1};
                for (int a = 0; a < 3; ++a) {
                  if (p[a] < 0) {
                    p[a] += bs;
                    e -= step[a];
                  } else if (p[a] >= bs) {
                    p[a] -= bs;
                    e += step[a];
                  }
                }
                if (around[e]) src = around[e][(p[0] * bs + p[1]) * bs + p[2]];
              }
              if (mismatch(here, src, j)) {
                bad.store(true, std::memory_order_relaxed);
                return;
              }
            }
          }
    }
  }, partGrain);
  return bad.load() ? one_writer_error(L) : HLB_OK;
}

void mark_inner_links(HostLattice& L) {
  L.inner.resize((size_t)L.N);
  parallel_ranges(L.N, [&](int, int64_t lo, int64_t hi) {
    for (int64_t k = lo; k < hi; ++k) {
      L.inner[(size_t)k] = 0;
      for (int d = 1; d < Q; ++d)
        if (link_of(L, k, d) != HLB_LINK_NONE &&
            L.site_at(L.coords[3 * k] + CX[d], L.coords[3 * k + 1] + CY[d], L.coords[3 * k + 2] + CZ[d]) >= 0)
          L.inner[(size_t)k] |= 1u << (d - 1);
    }
  });
}

void pull_table(const HostLattice& L, uint32_t* out) {
  const int64_t n = L.N;
  parallel_ranges(n, [&](int, int64_t lo, int64_t hi) {
    for (int64_t k = lo; k < hi; ++k) {
      const int64_t x = L.coords[3 * k], y = L.coords[3 * k + 1], z = L.coords[3 * k + 2];
      for (int j = 1; j < Q; ++j) {
        const bool plain = link_of(L, k, INV[j]) == HLB_LINK_NONE;
        out[(size_t)(j - 1) * n + k] = (uint32_t)(plain ? L.site_at(x - CX[j], y - CY[j], z - CZ[j]) : k);
      }
    }
  });
}

void push_table(const HostLattice& L, int64_t* out) {
  const int64_t n = L.N;
  for (int64_t k = 0; k < n; ++k) {
    const int64_t x = L.coords[3 * k], y = L.coords[3 * k + 1], z = L.coords[3 * k + 2];
    out[k * Q] = k * Q;
    for (int d = 1; d < Q; ++d) {
      const int64_t nb = L.site_at(x + CX[d], y + CY[d], z + CZ[d]);
      out[k * Q + d] = nb >= 0 ? nb * Q + d : n * Q;
    }
  }
}

}  // namespace hlb
