// lbm_kernels.h -- device-side data layout shared by the kernels and the
// host launcher.
//
// Slab layout.  The reference's LatticeData orders sites class-major
// (LatticeData.h:375-436); the host keeps that order for every API array.  On
// the device the site grid is cut into 8^3 bricks (occupied tiles in tile
// order, z fastest) and each brick into 8 slabs, one per block-local x; a
// slab's 64 lanes are its (y, z) positions, lane = y * 8 + z (the reference's
// in-block order, z fastest).  One wavefront handles one slab and a launch
// walks the list of slabs that hold at least one fluid site.  Storage is
// compact: the fluid lanes of a slab occupy consecutive slots from the slab's
// base in lane order (slot = base + number of fluid lanes below), bases
// rounded up to kSlabAlign slots.  (Measured on MI355X: 32-slot bases keep
// the read and write bytes at the layout's own size; 16-slot bases more
// than doubled both in the step kernels.)  A
// site's upstream neighbour is found arithmetically from the fluid masks and
// bases of the slabs around it, which the slab's record lists, so no
// per-site neighbour table is read.  A link whose upstream position is not
// fluid reads the site's own slot instead, which holds what a wall or iolet link
// hands back; a wall or iolet link to a position that is fluid (no thickness
// between two sites) is marked (kInnerLinks) and its value replaced by the
// boundary delegates.
//
// HBM layout (S = compact slots rounded up to 64):
//   A[2]   post-collision distributions, 19 planes of S (double, or float
//          g = f - w rho0 in the FP32-shifted form).
//   F      pre-collision staging of the same shape (initial state, uploads,
//          downloads).
//   rec    one 256-byte record per active slab (SlabRec).  Boundary sites
//          (collision classes 1-5) are numbered in slot order.
//   boundary arrays (NB boundary sites, stride SB): one BndRec, 18 planes of
//          float link distances, 3 planes of float wall normals.
//   iolet arrays (NI sites with iolet links, slot order, stride SI): 18 planes
//          of Ladd profile factors, and G, 19 planes of values the site's iolet
//          delegates computed for the next step where they cannot take the
//          place of a post-collision one (iolet_place).
#pragma once

#include <cstdint>

namespace hlb {

constexpr int kBrickSites = 512;  // positions per brick (8^3)
constexpr int kSlab = 64;         // positions per slab = lanes per wavefront
constexpr int kSlabAlign = 32;    // slab bases are multiples of this many slots
constexpr int kXcds = 8;          // accelerator complex dies on MI355X

// The slabs a lane can pull from: entries 0..8 are the slab's own x layer in
// the 3 x 3 bricks around it (index (dy+1)*3 + dz+1, 4 = the slab itself);
// 9..13 the layer at x - 1 and 14..18 the layer at x + 1 (in this brick or
// the next one in x), each in the brick itself, at dy -1, dy +1, dz -1,
// dz +1.  D3Q19 has no link with all three components nonzero, so no other
// slab is ever read.
constexpr int kReach = 19;
constexpr int reach_entry(int dx, int dy, int dz) {
  return dx == 0 ? (dy + 1) * 3 + (dz + 1)
                 : (dx < 0 ? 9 : 14) + (dy == 0 ? (dz == 0 ? 0 : (dz < 0 ? 3 : 4)) : (dy < 0 ? 1 : 2));
}

// One active slab: everything a wave needs before its first gather, in one
// 256-byte record read with scalar loads that do not wait on one another --
// the fluid masks and compact bases of the reachable slabs (a missing or
// empty slab has mask 0), the boundary-lane mask and the compact index of its
// first boundary lane.
struct SlabRec {
  uint64_t fm[kReach];    // fluid lanes of each reachable slab
  uint64_t bmask;         // boundary lanes of this slab
  int32_t base[kReach];   // first slot of each reachable slab
  int32_t bbase;          // boundary index of this slab's first boundary lane
  int32_t sid;            // brick * 8 + x (host bookkeeping)
  int32_t pad[3];
};
static_assert(sizeof(SlabRec) == 256, "slab record is four 64-byte scalar loads");

// One boundary site, for one 16-byte load issued ahead of the site's gathers.
// Bits are links (d - 1) or pull directions (j - 1); direction j's value is
// written by link INV[j].
struct BndRec {
  uint32_t far;    // directions BFL interpolates with the site's own value (q >= 1/2); kInnerLinks; bit 31: a wall site
  uint32_t near;   // directions BFL interpolates with the streamed value (q < 1/2); bits 18..: global iolet index
  uint32_t iolet;  // iolet links
  uint32_t ii;     // compact iolet index (sites with iolet links)
};
static_assert(sizeof(BndRec) == 16, "one 16-byte load");
constexpr uint32_t kLinkBits = (1u << 18) - 1u;
// Bit of BndRec::far at sites with a wall or iolet link to a fluid site (a wall of
// no thickness).  FP64 lattices without such links do no more than test the bit
// where BFL loads a site's own row, which cost nothing measurable.  In the FP32
// step any form of the test did on a 6k-site pipe, whose step is one chain of
// loads (6.6 us: 1.3 to 2.3%, a null pointer tested beside the GZS tables' 1.4%),
// so its kernels are compiled without it and once with it (inner_launch).
constexpr uint32_t kInnerLinks = 1u << 30;

// The brick tables of one lattice.
struct BrickTables {
  const SlabRec* rec;  // per active slab
  int64_t nslab;       // active slabs
};
constexpr int kMaxIolets = 256;  // iolets per lattice

// Launch shapes of the step kernels.  A shape is a workgroup tile of 2, 4 or
// 1 wavefronts (128, 256, 64 threads, one slab per wavefront, or two in FP32),
// a tile order and an occupancy level.
//   Tile orders: plain (workgroup w is tile w; the hardware hands workgroup w
//   to XCD w mod 8), XCD-contiguous (each XCD walks one contiguous eighth of
//   the tiles) and XCD chunks (chunks of kXcdChunk consecutive tiles dealt to
//   the XCDs in turn, so every XCD walks its own runs of neighbouring tiles
//   while all of them advance through the lattice together).
//   Levels 0..3 cap the waves resident per SIMD (none, 4, 3, 2) by giving
//   each workgroup dynamic LDS it does not use: fewer waves in flight keep
//   more of each wave's neighbour lines in the XCD's L2.  Levels 4 and 5
//   raise the floor instead: the kernel is compiled for at least 5/6 (FP64)
//   or 6/7 (FP32) waves per SIMD (fewer registers), for more loads in flight.
// Numbering (stable across builds):
//   0..35    shape (v % 6: 128 plain, 128 XCD, 256 plain, 256 XCD, 64 plain,
//            64 XCD) + 6 * level;
//   FP32 36..71: the same with two consecutive slabs per wavefront, both
//            slabs' gathers issued before either is waited for;
//   FP64 36..53, FP32 72..89: XCD chunks, block (u % 3: 128, 256, 64) +
//            3 * level, u = v - 36 (FP64) or v - 72 (FP32);
//   FP32 90..107: the same with two slabs per wavefront;
//   FP64 54..107 and FP32 108..215: FP64 0..53 and FP32 0..107 writing the
//            post-collision row with non-temporal stores (when the arrays are
//            far larger than the caches the next step will not find those
//            lines there anyway, and they no longer displace the lines the
//            gathers share; when the arrays fit the Infinity Cache they cost
//            the next step its hits).
constexpr int kShapeVariants = 36;  // plain and XCD-contiguous shapes x levels
constexpr int kChunkVariants = 18;  // XCD-chunk shapes x levels
constexpr int kFp64Shapes = kShapeVariants + kChunkVariants;  // per store policy
constexpr int kFp32Shapes = 2 * kFp64Shapes;                  // x slabs per wavefront
constexpr int kFp64Variants = 2 * kFp64Shapes;                // x store policy
constexpr int kFp32Variants = 2 * kFp32Shapes;
constexpr int kFp32DefaultVariant = 1;  // 128 slots (two slabs), XCD order, no cap (either form)
constexpr int kXcdChunk = 32;           // tiles per chunk in the XCD-chunk order
enum TileOrder { kOrderPlain = 0, kOrderXcd = 1, kOrderXcdChunks = 2 };
struct LaunchShape {
  int block;  // threads per workgroup tile
  int order;  // TileOrder
  int level;  // 0..5
  int spt;    // slabs per wavefront (1, or 2 in FP32)
  bool nt;    // non-temporal stores of the post-collision row
};
// The shape of a variant in range for its precision.
LaunchShape launch_shape(int variant, bool fp32);
inline int shape_slabs(const LaunchShape& l) { return l.block / kSlab * l.spt; }  // slabs per tile
// Workgroups to launch for `tiles` tiles: padded to a multiple of what the
// order's tile map covers (the padding tiles have no slab).
inline uint32_t shape_grid(const LaunchShape& l, int64_t tiles) {
  const int64_t mul = l.order == kOrderXcdChunks ? (int64_t)kXcds * kXcdChunk : (int64_t)kXcds;
  return (uint32_t)((tiles + mul - 1) / mul * mul);
}
unsigned shape_lds(const LaunchShape& l);  // dynamic LDS bytes per workgroup

// The variant a lattice or batch reports until one is set or autotuned: the
// default, or its non-temporal twin once its distributions (two sets of 19
// planes) exceed the 256 MB Infinity Cache.
constexpr int64_t kInfinityCacheBytes = int64_t(256) << 20;
inline int64_t distribution_bytes(int64_t S, bool fp32) { return 2 * 19 * (fp32 ? 4 : 8) * S; }
inline int default_variant(int64_t dist_bytes, bool fp32) {
  const bool nt = dist_bytes > kInfinityCacheBytes;
  return kFp32DefaultVariant + (nt ? (fp32 ? kFp32Shapes : kFp64Shapes) : 0);
}

// The shape it is launched in meanwhile, by where its distributions live.
//   In the Infinity Cache: one-slab tiles in XCD order, cached stores (variant
//   5).  Against the two-slab tiles of variant 1 a step of the 30k-site
//   cylinder takes 5.75 instead of 6.4 us (its 480 waves reach more CUs), of a
//   6k-site pipe 6.6 / 7.0, of the 0.70M-site Y-bifurcation the same (FP64
//   45.3 / 45.6, FP32 27.1 / 27.3).
//   Beyond it: non-temporal row stores; up to 2.5 caches the two-slab tiles in
//   XCD order (0.58 GB FP64 pipe 110.9 us against 116.6 in chunks, 289 MB FP32
//   pipe 58.6 / 61.1; 0.50 GB bifurcation the other way, 112.7 / 105.9), above
//   that one-slab tiles in XCD chunks, which keep all XCDs within a few chunks
//   of one another, so that lines shared across a chunk's edge are still in
//   the Infinity Cache (XCD order / chunks: 0.70 GB FP32 tree 174 / 159 us, 1.5
//   GB FP64 pipe 307 / 293, 1.0 GB FP32 pipe 290 / 233, 2.7 GB FP64 tree 604 /
//   563, 2.5 GB FP64 bifurcation 522 / 508).  A batch takes the chunks from the
//   cache's size on: a chunk's edge cuts few of its small members (20 pipes,
//   0.29 GB: 73.1 / 67.8 us).
inline int default_launch(int64_t dist_bytes, bool fp32, bool batch = false) {
  const int chunk64 = (fp32 ? 2 * kShapeVariants : kShapeVariants) + 2;
  if (dist_bytes <= kInfinityCacheBytes) return 5;
  const bool chunks = batch || dist_bytes > kInfinityCacheBytes * 5 / 2;
  return (fp32 ? kFp32Shapes : kFp64Shapes) + (chunks ? chunk64 : 1);
}

// The FP32 variant launched in place of `variant` when a lattice or a member of a
// batch has links between fluid sites: one-slab tiles in XCD order with its store
// policy, the one shape compiled for them.
inline int inner_launch(int variant) { return (launch_shape(variant, true).nt ? kFp32Shapes : 0) + 5; }

// Guo-Zheng-Shi wall links (GuoZhengShiDelegate.h:123-294).  Sites whose
// pre-collision f the link kernel needs (GZS wall sites and the next fluid
// site out along a link) store it in P during the step; the link kernel
// then forms each GZS link's value for the next step in GW.
struct GzsTables {
  const uint64_t* pmask;  // per active slab: lanes that store their pre-collision f
  const int32_t* pbase;   // per active slab: P index of the first such lane
  const uint32_t* bgz;    // per boundary site: wall links whose value comes from GW
  const int32_t* bgzbase; // per boundary site: GW index of its first GZS link
  const uint32_t* inner;  // per boundary site: wall and iolet links to a fluid site (any wall delegate; see kInnerLinks)
  int64_t SP;             // P plane stride
};

struct GzsLink {
  int32_t site_p;   // P index of the wall site
  int32_t nb_p;     // P index of the next site out (regular branch), else -1
  int32_t dir;      // wall link direction d (the value goes to INV[d])
  int32_t mode;     // 1: this site only, 2: with the next site out, 3: velocity iolet beyond
  int32_t gi;       // global iolet index (mode 3)
  float q;          // wall distance as stored
  double s, s2;     // iolet profile factors at x + c_INV[d] (mode 3): speed = vmax s + vmax2 s2
};

// Windkessel state of one iolet (InOutLetWK2.cc:13-18, InOutLetWK3.cc:13-18)
// plus its constants; updated on the device between steps.
struct WkIolet {
  double density, densityNew, flowRate, flowRateOld, flowRateNew, siteCount;
  double area, resistance, r_c, r_p, capacitance;
  int32_t kind;            // HLB_IOLET_WK2 / HLB_IOLET_WK3, anything else: not a Windkessel
  int32_t centre_coupled;  // the centre site is one of this iolet's coupling sites
  int32_t list_begin, list_end;  // the iolet's coupling sites: positions in the coupling order
};

// A Windkessel iolet as the per-step kernels see it: its state and the
// buffers of the lattice it belongs to.  Arrays of these let one launch
// serve the Windkessel iolets of every lattice in a batch.
struct WkRef {
  WkIolet* w;
  double* io_dens;        // the lattice's rows of per-step values, ghost densities first
  const double* contrib;  // the lattice's u.(-n) terms in the coupling order, even steps' and odd steps'
  int64_t stride;         // from the first to the second
  int32_t g, row;         // iolet index in its lattice, row stride
  int32_t ordered;        // 1: sum in the reference's site order (FP64 form); 0: tree (FP32-shifted form)
  int32_t pad_;
};

// The Windkessel share of a launch (windkessel.h): its first `groups`
// workgroups (a multiple of the XCD count), one of which serves each iolet.
struct WkLaunch {
  const WkRef* refs;
  int32_t n;
  uint32_t groups;
  int32_t steps;  // of the sequence
  int32_t pad_;
};
inline WkLaunch wk_launch(const WkRef* refs, int n, int64_t steps) {
  return WkLaunch{refs, n, (uint32_t)((n + kXcds - 1) / kXcds * kXcds), (int32_t)steps, 0};
}

struct StepArgs {
  // Per-plane base pointers, passed as separate scalars so each access is one
  // SGPR base plus a 32-bit VGPR offset.
  const double* ain[19];
  double* aout[19];
  BrickTables bt;
  const BndRec* __restrict__ bnd;  // global iolet index: inlets 0..n_in-1, outlets follow
  const float* __restrict__ bq;
  const float* __restrict__ bnrm;
  double* __restrict__ G;
  const double* __restrict__ ladd_s;   // 18 planes of SI: velocity profile factor per iolet link
  const double* __restrict__ ladd_s2;  // 18 planes of SI: second factor (Womersley), else 0
  double* __restrict__ rho;
  double* __restrict__ u;
  double* __restrict__ wss;
  const double* __restrict__ io_n;    // 3 per iolet: the normal in double (Ladd)
  const double* __restrict__ io_dens; // this step's ghost density per iolet
  const double* __restrict__ io_vmax; // this step's peak speed per iolet (Womersley: cos wt)
  const double* __restrict__ io_vmax2; // this step's second speed factor (Womersley: sin wt), else 0
  const uint32_t* __restrict__ wk_bit; // per iolet: the link bit of its Windkessel coupling direction
  const int32_t* __restrict__ wk_pos;  // per iolet site: its place in the coupling order (coupling sites only)
  double* __restrict__ wk_contrib;     // u.(-n) of this step per coupling site, in the coupling order
  int64_t N, S, SB, SI;
  int32_t n_in;
  int32_t inlet_bc;
  int32_t outlet_bc;
  double tau;         // LbmParameters tau
  double omega;       // -1/tau
  double half_omega;  // 0.5*omega (TRT)
  double half_omega_minus;
  double les_k;       // 18 sqrt(2) C_s^2 evaluated in the reference's order
  int32_t general_gather;  // 1: the steady step takes the general gather on any lattice
  int32_t step;            // of the sequence
  WkLaunch wk;
  // LES sponge layer: vTau per slot (nullptr: none), this step's time (t
  // while t < lifetime, else -1), lifetime / 2 (integer division) and lifetime.
  const double* __restrict__ vtau;
  const double* __restrict__ sp_t;
  double sp_half, sp_life;
  GzsTables gz;       // pmask == nullptr: no GZS walls
  double* P;
  const double* GW;
};

// One lattice of the FP32-shifted form.  The storage holds g = f - w rho0
// (rho0 = 1) in float; a launch advances every member of a table, one
// workgroup tile of 256 device slots at a time, so a single lattice and a
// batch of lattices of uneven size run the same kernel.  Layout per member is
// the FP64 one with float planes for A, F and G.
struct Member32 {
  float* A[2];            // post-collision g, 19 planes of S
  const float* F;         // pre-collision g (initial state / checkpoint)
  BrickTables bt;
  const BndRec* bnd;
  const float* bq;
  const float* bnrm;
  float* G;               // 19 planes of SI (see iolet_place)
  const double* ladd_s;
  const double* ladd_s2;
  double* rho;
  double* u;
  double* wss;
  const float* io_nf;
  const double* io_n;
  const double* io_dens;  // one value per iolet, a row per step of the launch sequence
  const double* io_vmax;
  const double* io_vmax2;
  const uint32_t* wk_bit;
  const int32_t* wk_pos;
  double* wk_contrib;     // even steps' terms, then wk_stride on the odd steps'
  int64_t wk_stride;
  int64_t N, S, SB, SI;
  int32_t row, n_in;      // row stride of the per-step values
  int32_t kernel, inlet_bc, outlet_bc;
  int32_t cur0;           // A[cur0] holds the latest values when the sequence starts
  int32_t first0;         // 1: step 0 of the sequence reads F (pre-collision)
  int32_t props_at;       // step of the sequence that writes rho, u, WSS (-1: none)
  uint32_t wg_begin;      // first workgroup tile of this member in the launch (tiles of whole slabs)
  float tau, omega, half_omega, half_omega_minus, les_k;
  int32_t pad_;
  GzsTables gz;           // pmask == nullptr: no GZS walls
  float* P;
  const float* GW;
  const float* vtau;      // LES sponge layer (see StepArgs); nullptr: none
  const double* sp_t;     // one value, a row per step of the launch sequence
  double sp_half, sp_life;
};

}  // namespace hlb
