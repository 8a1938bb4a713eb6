// handle.h -- the handle behind hlb_handle and the internals the single
// lattice and batch entry points share.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/hemepure_amd.h"
#include "errors.h"
#include "lattice.h"
#include "lbm_kernels.h"
#include "transfer.h"

namespace hlb {

hipError_t launch_step_fp64(const StepArgs& a, int kernel, bool first, bool props, int variant, hipStream_t s);
hipError_t launch_gzs_fp64(const StepArgs& a, int kernel, const GzsLink* links, int n, const double* vmax,
                           double* GW, hipStream_t s);
hipError_t launch_gzs_fp32(const Member32* members, const GzsLink* links, int n, int step, hipStream_t s);
hipError_t launch_upstream_table(const BrickTables& bt, uint32_t* out, int64_t S, hipStream_t s);
size_t monitor_scratch(int64_t nslab);
hipError_t launch_monitor(const BrickTables& bt, const double* rho, const double* u, int64_t S, void* scratch,
                          double* out, bool signal, hipStream_t s);
hipError_t launch_gather_fp64(const StepArgs& a, double* F, int64_t S, hipStream_t s);
hipError_t launch_stress_fp64(const StepArgs& a, int kernel, const void* F, bool fp32, double* out, hipStream_t s);
hipError_t launch_fill_fp64(double* F, int64_t N, int64_t S, const double* vals, hipStream_t s);
hipError_t launch_unstable_fp64(const BrickTables& bt, const double* F, int64_t S, int* flag, hipStream_t s);
hipError_t launch_wk_start(const WkRef* refs, int n, hipStream_t s);
hipError_t launch_wk_flush(const WkRef* refs, int n, int last, hipStream_t s);
hipError_t launch_step_fp32(const Member32* members, const int32_t* wg_member, uint32_t grid, int step,
                            const WkLaunch& wk, int variant, bool inner, hipStream_t s);
hipError_t launch_gather_fp32(const Member32* members, int64_t nslab, float* F, hipStream_t s);
hipError_t launch_fill_fp32(float* F, int64_t N, int64_t S, const float* vals, hipStream_t s);
hipError_t launch_unstable_fp32(const BrickTables& bt, const float* F, int64_t S, int* flag, hipStream_t s);
hipError_t launch_cycle_delta(const double* u, float* prev, int64_t N, int64_t S, unsigned* out_bits,
                              hipStream_t s);



inline constexpr double kPi = 3.14159265358979323846264338327950288;  // src/constants.h:17
inline constexpr int64_t kChunk = 1024;  // steps of iolet values staged per upload

inline constexpr int64_t kStageHead = 64;  // doubles ahead of them for the FP32 form's member record
inline constexpr int64_t kStageResult = 56;  // where the pinned staging's head takes the monitors' results
static_assert(sizeof(Member32) <= sizeof(double) * kStageResult, "the record fits the staging's head");

// Whether a sequence of n one-launch steps over nslab slabs is replayed from a
// captured graph rather than launched step by step.  A replay costs ~20 us to
// start and, the first time, ~4 us a step to capture; a launch from the host
// costs ~2.4 us, hidden behind the step before it, and ~0.6 us more between
// kernels, which shows only while steps take a few us.  Graph / eager, us for n
// steps (FP64): 6.5k sites n = 8 68 / 67, n = 16 111 / 117, n = 300 1636 / 1880;
// 30k sites n = 16 120 / 124, n = 300 1801 / 2021; 67k sites (~1.4k slabs) n =
// 16 159 / 153, n = 300 2443 / 2541; 127k sites (~2.5k slabs) n = 16 197 / 190,
// n = 300 3208 / 3218; 430k sites n = 8 226 / 217, n = 300 7471 / 7468.
inline constexpr int64_t kReplaySteps = 16;
inline bool replay_pays(int64_t n, int64_t nslab) { return n >= kReplaySteps && nslab <= 2048; }

inline int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

struct HostIolet {
  hlb_iolet_desc d;
  double n[3];    // InOutLet::SetNormal: normalised in double (InOutLet.h:169-172)
  float nf[3];    // the Vector3D<float> copy Nash uses (NashZerothOrderPressureDelegate.h:57-58)
  std::vector<double> table;
  double minSimDensity = 1.0;
  int dirs0 = 0;               // direction closest to the normal (coupling direction)
  int64_t centre = -1;         // centre site, reference order (BoundaryValues.cc:109-128)
  bool centreCoupled = false;
  bool IsWK() const { return d.kind == HLB_IOLET_WK2 || d.kind == HLB_IOLET_WK3; }
  bool IsVelocity() const {
    return d.kind == HLB_IOLET_PARABOLIC || d.kind == HLB_IOLET_FILEVEL || d.kind == HLB_IOLET_WOMERSLEY;
  }
};

template <typename T>
struct DevBuf {
  T* p = nullptr;
  size_t n = 0;
  bool owned = true;  // false: a part of another allocation
  DevBuf() = default;
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  ~DevBuf() { release(); }
  void release() {
    if (p && owned) (void)hipFree(p);
    p = nullptr;
    owned = true;
  }
  hipError_t alloc(size_t count) {
    release();
    n = count;
    if (count == 0) return hipSuccess;
    return hipMalloc(&p, sizeof(T) * count);
  }
  void view(void* part, size_t count) {
    release();
    p = static_cast<T*>(part);
    n = count;
    owned = false;
  }
};

// Device arrays made together: those up to kPackBytes are laid out in one
// allocation and filled with one copy (an allocation costs ~11 us, its release
// ~29 us and a blocking copy ~46 us whatever their size), larger ones get their
// own.  add() keeps a pointer to `data` (null: zeros) until commit().
class DevPack {
 public:
  template <typename T>
  void add(DevBuf<T>& buf, const T* data, size_t count) {
    items_.push_back({&buf, data, sizeof(T), count, [](void* b, void* part, size_t n) {
                        auto* d = static_cast<DevBuf<T>*>(b);
                        if (part) {
                          d->view(part, n);
                          return hipSuccess;
                        }
                        return d->alloc(n);
                      },
                      [](void* b) { return (void*)static_cast<DevBuf<T>*>(b)->p; }});
  }
  template <typename T>
  void add(DevBuf<T>& buf, const std::vector<T>& data) {
    add(buf, data.data(), data.size());
  }
  // Allocates and fills everything (zeros asynchronously on s).
  hipError_t commit(DevBuf<char>& arena, hipStream_t s);

 private:
  static constexpr size_t kPackBytes = size_t(1) << 20, kAlign = 256;
  struct Item {
    void* buf;
    const void* data;
    size_t size, count;
    hipError_t (*place)(void*, void*, size_t);
    void* (*where)(void*);
  };
  std::vector<Item> items_;
};

// Blocking copy in s's order.  Not hipMemcpy: that runs on the legacy stream, which
// fails, and breaks the capture, while any other thread captures a graph.
inline hipError_t copy_now(void* dst, const void* src, size_t bytes, hipMemcpyKind kind, hipStream_t s) {
  const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
  return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

inline int dev_fail(hipError_t e, const char* what) {
  return fail(HLB_EDEVICE, std::string(what) + ": " + hipGetErrorString(e));
}

#define HLB_CHECK(expr)                                 \
  do {                                                  \
    hipError_t _e = (expr);                             \
    if (_e != hipSuccess) return dev_fail(_e, #expr);   \
  } while (0)

}  // namespace hlb

struct hlb_lattice {
  hlb::DevBuf<char> arena, fields_mem, a_mem;  // what the arrays below are parts of
  hlb::HostLattice L;
  hlb_params params{};
  std::vector<hlb::HostIolet> iolets;  // inlets then outlets
  int n_in = 0, n_out = 0;
  int device = 0;
  hlb::HostLane lane;  // the stream, events and pinned staging below, while there is a device state
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  void use_lane() {
    stream = lane.stream;
    ev0 = lane.ev0;
    ev1 = lane.ev1;
    h_stage = lane.stage;
  }
  // Device slots (compact slab layout): perm[slot] = reference index or -1
  // for padding, inv[k] = slot of reference index k.
  std::vector<int32_t> perm, inv;
  int64_t nbrick = 0, nslab = 0;
  int slab_order = HLB_ORDER_TILE;  // HLB_ORDER_TILE or HLB_ORDER_LAYER, fixed at create
  std::vector<int32_t> h_slab, h_sbase;  // per active slab: brick * 8 + x, first slot
  std::vector<uint64_t> h_fmask;          // per active slab: fluid lanes
  std::vector<hlb::SlabRec> h_rec;        // the records the kernels read
  // Boundary sites (classes 1-5) and iolet sites in device order.
  std::vector<int32_t> bsite;  // reference index of boundary slot b
  std::vector<int32_t> isite;  // reference index of iolet slot i
  int64_t S = 0, NB = 0, SB = 0, NI = 0, SI = 0;
  hlb::DevBuf<double> A[2], F, G, ladd_s, rho, u, wss, io_n, feq_vals;
  hlb::DevBuf<hlb::BndRec> bnd;  // boundary records
  hlb::DevBuf<hlb::SlabRec> rec;  // slab records
  hlb::DevBuf<float> bq, bnrm, io_nf;
  hlb::DevBuf<int32_t> dinv;      // inv on the device (transfer.hip)
  // Guo-Zheng-Shi walls (params.wall_bc == HLB_WALL_GZS).
  std::vector<hlb::GzsLink> gz_links_host;
  std::vector<uint64_t> h_pmask;
  std::vector<int32_t> h_pbase, h_bgz, h_bgzbase;
  int64_t NP = 0, SP = 0;
  hlb::DevBuf<hlb::GzsLink> gz_links;
  hlb::DevBuf<uint64_t> pmask;
  hlb::DevBuf<int32_t> pbase, bgzbase;
  hlb::DevBuf<uint32_t> bgz, inner;  // inner: L.inner per boundary site
  hlb::DevBuf<double> P64, GW64;
  hlb::DevBuf<float> P32, GW32;
  hlb::DevBuf<char> mon_scratch;  // monitor partials, allocated on first use
  hlb::DevBuf<double> stress;     // 17 stress planes, allocated on first use
  // FP32-shifted storage (params.precision == HLB_FP32_SHIFTED): float A, F, G.
  hlb::DevBuf<float> A32[2], F32, G32, feq32;
  // Windkessel iolets: device state, coupling bit per iolet, per-site terms,
  // coupling sites per iolet in the reference's site order.
  bool any_wk = false;
  std::vector<int32_t> wk_list;
  std::vector<hlb::WkIolet> wk_host;
  hlb::DevBuf<hlb::WkIolet> wk;
  hlb::DevBuf<uint32_t> wk_bit;
  hlb::DevBuf<double> wk_contrib;  // two buffers of wk_stride() terms, even and odd steps'
  int64_t wk_stride() const { return (int64_t)(wk_list.empty() ? 1 : wk_list.size()); }
  hlb::DevBuf<int32_t> wk_pos;  // per iolet site: its place in wk_list (coupling sites), else -1
  std::vector<hlb::WkRef> wk_refs_host;  // one per Windkessel iolet
  hlb::DevBuf<hlb::WkRef> wk_refs;
  struct hlb_batch* batch = nullptr;     // the batch this lattice belongs to, if any
  // LES sponge layer (hlb_set_sponge; LBGKLESSpongeLayer.h:87-148): vTau per
  // device slot, the lifetime in steps (0: none, pure LES) and the per-step
  // time rows the kernels read (t while t < lifetime, else -1).
  int64_t sponge_life = 0;
  double sponge_ratio = 1.0, sponge_width = 0.0;
  std::vector<double> h_vtau;
  hlb::DevBuf<double> vtau64;
  hlb::DevBuf<float> vtau32;
  // What a sequence of steps reads from the host, and its pinned staging: the
  // one-member table the FP32 kernel reads (kStageHead doubles), then a row per
  // step (per iolet the ghost density, then the two speed factors, then the
  // sponge's time).
  hlb::DevBuf<double> stage;
  double* h_stage = nullptr;
  // Nothing queued reads the staging: set when a monitor's result has arrived,
  // cleared where the staging is written.
  bool staging_idle = false;
  int iolet_count() const { return iolets.empty() ? 1 : (int)iolets.size(); }
  int64_t row() const { return 3 * (int64_t)iolet_count() + 1; }
  int64_t stage_doubles() const { return hlb::kStageHead + hlb::kChunk * row(); }
  double* rows() const { return stage.p + hlb::kStageHead; }
  // Whether an n-step sequence reads its rows from the pinned staging itself: a
  // single FP64 step, where only the iolet layers' waves read them (once, over
  // the bus) and no Windkessel iolet writes them.  On a 14k-site pipe a step
  // and the wait for it take 20.1 us so, 22.6 with the copy.
  bool rows_in_place(int64_t n) const { return n == 1 && !fp32() && wk_refs_host.empty() && sponge_life == 0; }
  // Pinned doubles the monitors' kernels write their results to.
  double* result() const { return h_stage + hlb::kStageResult; }
  hlb::Member32* member() const { return reinterpret_cast<hlb::Member32*>(stage.p); }
  int cur = 0;                // A[cur] holds the latest post-collision values
  bool have_post = false;     // false: the next step reads the pre-collision F
  bool f_valid = false;
  int64_t t = 1;              // 1-indexed step that runs next
  double omega = 0, half_omega = 0, half_omega_minus = 0, les_k = 0;
  std::vector<double> h_ladd_s;  // Ladd profile factors, 2 x 18 planes of SI, device iolet order
  bool device_ready = false;
  bool iolets_set = false;   // hlb_create with params, or hlb_set_iolets
  int variant = hlb::kFp32DefaultVariant;  // launch shape of the steady-state step, as reported
  bool variant_chosen = false;              // set by hlb_set_variant / hlb_autotune; else default_variant
  // The variant steps are launched in.
  int launch_variant() const {
    const int v = variant_chosen ? variant : hlb::default_launch(hlb::distribution_bytes(S, fp32()), fp32());
    return fp32() && inner_links() ? hlb::inner_launch(v) : v;
  }
  bool inner_links() const { return !L.inner.empty(); }  // links between fluid sites
  bool general_gather = false;  // HLB_FP64_GENERAL_GATHER=1 when the device state was made
  // Step sequences captured into HIP graphs and replayed: one per (length,
  // property flag, first-step flag, buffer parity, launch shape); the FP32
  // form reads the last two from its member record, so they are 0 there.
  struct StepGraph {
    int64_t n;
    int props, first, cur, variant;
    hipGraphExec_t exec;
  };
  std::vector<StepGraph> graphs;
  bool use_graph = true;
  // GZS walls add a launch per step, which a replay saves at any size.
  bool replays(int64_t n) const { return hlb::replay_pays(n, gz_links_host.empty() ? nslab : 0); }
  void drop_graphs() {
    for (StepGraph& g : graphs) (void)hipGraphExecDestroy(g.exec);
    graphs.clear();
  }

  ~hlb_lattice() {
    if (stream) {
      (void)hipStreamSynchronize(stream);
      drop_graphs();
    }
    hlb::give_lane(lane);
    if (device_ready) hlb::transfer_close();
  }
  bool fp32() const { return params.precision == HLB_FP32_SHIFTED; }
  hlb::GzsTables gz_tables() const {
    const uint32_t* in = inner_links() ? inner.p : nullptr;
    if (gz_links_host.empty()) return hlb::GzsTables{nullptr, nullptr, nullptr, nullptr, in, 0};
    return hlb::GzsTables{pmask.p, pbase.p, bgz.p, bgzbase.p, in, SP};
  }
  hlb::BrickTables tables() const {
    return hlb::BrickTables{rec.p, nslab};
  }
};

namespace hlb {

// Shared by the single-lattice and batch entry points (capi.hip).
int ensure_device(hlb_lattice* h);
int stage_iolet_values(hlb_lattice* h, int64_t t, int64_t n, hipStream_t s);
Member32 member_record(const hlb_lattice* h, int props_at);
// The lattice state after an n-step sequence (A parity, first-step flag, time).
void advance_state(hlb_lattice* h, int64_t n);
// Removes a lattice that is being destroyed from its batch (batch.hip).
void batch_forget(struct hlb_batch* b, hlb_lattice* h);
// Device bytes a lattice holds once it has a state (capi.hip).
int64_t device_bytes(const hlb_lattice* h);
// The stream a batch's launches run on (batch.hip).
hipStream_t batch_stream(struct hlb_batch* b);

}  // namespace hlb
