// transfer.hip -- site arrays between the device's slot order and the
// caller's host arrays in the reference's site order.
//
// The callers of hlb_get_fields, hlb_download_f, hlb_get_stress and
// hlb_upload_f hold pageable arrays of site records (W doubles per site in the
// reference's class-major order), the device holds W planes in slot order.
// Both the reordering and the transposition run on the GPU: export_sites
// gathers the planes through the site -> slot index straight into pinned host
// memory (whole contiguous runs, so the bus sees full lines), import_sites
// reads such a chunk and scatters it.  Chunks of one slot (kSlotBytes) are
// taken by a few host threads, each with two slots: while the GPU fills one,
// the thread copies the other into the caller's array, which is where its
// pages are first touched.  What bounds a large transfer is that host copy
// (page faults included) and the bus, no longer one thread that walks an index
// over strided planes.  Measured on MI355X, one pass before and after: 304 MB
// of fields of a 7.6M-site FP32 tree 85 -> about 8 ms, distributions saved and
// restored for 0.42M FP64 sites (2 x 63 MB) 20 -> 4 ms, their 57 MB of stress
// rows 18 -> 1.5 ms, fields of a 30k-site cylinder 0.14 -> 0.07 ms.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "device_util.h"
#include "errors.h"
#include "handle.h"
#include "transfer.h"

namespace hlb {

namespace {

constexpr size_t kSlotBytes = size_t(1) << 20;
constexpr int kMaxWorkers = 8;                 // host threads of one transfer
constexpr int kPoolSlots = 2 * kMaxWorkers;    // slots kept between transfers, per process
// Up to here the calling thread copies alone (3.4 MB of fields 0.19 ms so, 0.32
// on four threads with smaller chunks).
constexpr size_t kInlineBytes = size_t(3) << 20;

// ---- pinned chunks ----------------------------------------------------------

struct Slot {
  char* p = nullptr;
  hipEvent_t ev = nullptr;  // the last kernel that used the slot
  int device = -1;
};

// Slots outlive a transfer (pinning a page costs more than copying it) and
// lanes a lattice, but not the last lattice with a device state or server of
// the process.
struct Pool {
  std::mutex mu;
  std::vector<Slot> idle;
  std::vector<HostLane> lanes;
  int users = 0;
};
constexpr size_t kIdleLanes = 16;
constexpr size_t kIdleLaneDoubles = size_t(1) << 18;  // staging beyond 2 MiB is not kept

Pool& pool() {
  static Pool* p = new Pool;  // never destroyed: the HIP runtime may be gone at exit
  return *p;
}

void free_slot(Slot& s) {
  if (s.ev) (void)hipEventDestroy(s.ev);
  if (s.p) (void)hipHostFree(s.p);
  s = Slot{};
}

int take_slot(int device, Slot& out) {
  {
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.mu);
    for (size_t i = 0; i < P.idle.size(); ++i)
      if (P.idle[i].device == device) {
        out = P.idle[i];
        P.idle.erase(P.idle.begin() + (std::ptrdiff_t)i);
        return HLB_OK;
      }
  }
  Slot s;
  s.device = device;
  hipError_t e = hipHostMalloc((void**)&s.p, kSlotBytes, hipHostMallocDefault);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&s.ev, hipEventDisableTiming);
  if (e != hipSuccess) {
    free_slot(s);
    return dev_fail(e, "hipHostMalloc(transfer chunk)");
  }
  out = s;
  return HLB_OK;
}

void give_slot(Slot& s) {
  if (!s.p) return;
  Pool& P = pool();
  std::unique_lock<std::mutex> lk(P.mu);
  if (P.users > 0 && P.idle.size() < (size_t)kPoolSlots) {
    P.idle.push_back(s);
    s = Slot{};
    return;
  }
  lk.unlock();
  free_slot(s);
}

// ---- kernels ----------------------------------------------------------------

// One array of a chunk: `planes` planes of slot order, to or from element
// `at` of the chunk on.
struct ChunkPart {
  const void* src;
  int32_t planes;
  int32_t at;
};
struct Chunk {
  ChunkPart part[kMaxTransferParts];
  const int32_t* slot;  // slot of the chunk's first site, then one per site
  int64_t S;
  int32_t n;            // sites of the chunk
};

template <int W>
__device__ __forceinline__ void split(uint32_t e, uint32_t& k, uint32_t& c) {
  k = e / W;
  c = e - k * W;
}

// Element e of a part is component c of site k (consecutive lanes write
// consecutive elements).
template <typename T>
__global__ __launch_bounds__(kBlock) void export_chunk(Chunk a, double* __restrict__ out) {
  const ChunkPart p = a.part[blockIdx.y];
  const uint32_t total = (uint32_t)(a.n * p.planes);
  for (uint32_t e = blockIdx.x * kBlock + threadIdx.x; e < total; e += gridDim.x * kBlock) {
    uint32_t k = e, c = 0;
    switch (p.planes) {
      case 1: break;
      case 3: split<3>(e, k, c); break;
      case 6: split<6>(e, k, c); break;
      case 17: split<17>(e, k, c); break;
      default: split<Q>(e, k, c); break;
    }
    const T v = static_cast<const T*>(p.src)[(int64_t)c * a.S + a.slot[k]];
    // float planes are the shifted distributions g = f - w
    out[p.at + e] = sizeof(T) == 8 ? (double)v : (double)v + Wt((int)c);
  }
}

template <typename T>
__global__ __launch_bounds__(kBlock) void import_chunk(const double* __restrict__ in, const int32_t* __restrict__ slot,
                                                       int32_t n, int64_t S, T* __restrict__ out) {
  const uint32_t total = (uint32_t)n * Q;
  for (uint32_t e = blockIdx.x * kBlock + threadIdx.x; e < total; e += gridDim.x * kBlock) {
    uint32_t k, c;
    split<Q>(e, k, c);
    const double v = in[e];
    out[(int64_t)c * S + slot[k]] = sizeof(T) == 8 ? (T)v : (T)(v - Wt((int)c));
  }
}

uint32_t blocks_for(int64_t elements) {
  return (uint32_t)std::max<int64_t>(1, std::min<int64_t>((elements + kBlock - 1) / kBlock, 1024));
}

// ---- the chunk loop ---------------------------------------------------------

// Takes every chunk through start(slot, chunk), which queues its kernel on the
// handle's stream, and, once that kernel has run, finish(slot, chunk), on up
// to kMaxWorkers threads that each alternate between two slots.
template <typename Start, typename Finish>
int run_chunks(hlb_lattice* h, int64_t chunks, size_t bytes, Start&& start, Finish&& finish) {
  std::atomic<int64_t> next{0};
  std::atomic<bool> stop{false};
  const int nw = bytes <= kInlineBytes ? 1 : (int)std::min<int64_t>(kMaxWorkers, (chunks + 1) / 2);
  std::vector<int> rcs((size_t)nw, HLB_OK);
  std::vector<std::string> msgs((size_t)nw);
  auto work = [&](int w) {
    Slot s[2];
    int64_t in_slot[2] = {-1, -1};
    auto settle = [&](int i) -> int {
      if (in_slot[i] < 0) return HLB_OK;
      HLB_CHECK(hipEventSynchronize(s[i].ev));
      finish(s[i].p, in_slot[i]);
      in_slot[i] = -1;
      return HLB_OK;
    };
    auto body = [&]() -> int {
      HLB_CHECK(hipSetDevice(h->device));
      for (int i = 0;; i ^= 1) {
        const int64_t c = next.fetch_add(1);
        if (c >= chunks || stop.load()) break;
        int rc = s[i].p ? settle(i) : take_slot(h->device, s[i]);
        if (rc != HLB_OK) return rc;
        rc = start(s[i].p, c);
        if (rc != HLB_OK) return rc;
        in_slot[i] = c;
        HLB_CHECK(hipEventRecord(s[i].ev, h->stream));
      }
      int rc = settle(0);
      if (rc == HLB_OK) rc = settle(1);
      return rc;
    };
    rcs[(size_t)w] = body();
    if (rcs[(size_t)w] != HLB_OK) {
      msgs[(size_t)w] = last_error();
      stop.store(true);
      (void)hipStreamSynchronize(h->stream);  // no kernel may still use a slot that goes back
    }
    give_slot(s[0]);
    give_slot(s[1]);
  };
  std::vector<std::thread> threads;
  threads.reserve((size_t)nw);
  for (int w = 1; w < nw; ++w) {
    try {
      threads.emplace_back(work, w);
    } catch (const std::exception&) {
      break;  // fewer threads: the chunks are taken by those there are
    }
  }
  int device = -1;
  const bool known = hipGetDevice(&device) == hipSuccess;
  work(0);
  for (std::thread& t : threads) t.join();
  if (known && device != h->device) (void)hipSetDevice(device);
  for (int w = 0; w < nw; ++w)
    if (rcs[(size_t)w] != HLB_OK) return fail(rcs[(size_t)w], msgs[(size_t)w]);
  return HLB_OK;
}

}  // namespace

namespace {

void free_lane(HostLane& l) {
  if (l.stream) (void)hipStreamDestroy(l.stream);
  if (l.ev0) (void)hipEventDestroy(l.ev0);
  if (l.ev1) (void)hipEventDestroy(l.ev1);
  if (l.stage) (void)hipHostFree(l.stage);
  l = HostLane{};
}

}  // namespace

int take_lane(int device, size_t doubles, HostLane& out) {
  {
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.mu);
    for (size_t i = 0; i < P.lanes.size(); ++i)
      if (P.lanes[i].device == device && P.lanes[i].doubles >= doubles) {
        out = P.lanes[i];
        P.lanes.erase(P.lanes.begin() + (std::ptrdiff_t)i);
        return HLB_OK;
      }
  }
  HostLane l;
  l.device = device;
  l.doubles = doubles;
  hipError_t e = hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipEventCreate(&l.ev0);
  if (e == hipSuccess) e = hipEventCreate(&l.ev1);
  if (e == hipSuccess) e = hipHostMalloc((void**)&l.stage, sizeof(double) * doubles, hipHostMallocDefault);
  if (e != hipSuccess) {
    free_lane(l);
    return dev_fail(e, "stream and staging of a lattice");
  }
  out = l;
  return HLB_OK;
}

void give_lane(HostLane& lane) {
  if (!lane.stream) return;
  // a stream whose capture went wrong would fail in the lattice that gets it next
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  const bool usable = hipStreamIsCapturing(lane.stream, &status) == hipSuccess && status == hipStreamCaptureStatusNone &&
                      hipStreamQuery(lane.stream) == hipSuccess;
  Pool& P = pool();
  std::unique_lock<std::mutex> lk(P.mu);
  if (usable && P.users > 0 && P.lanes.size() < kIdleLanes && lane.doubles <= kIdleLaneDoubles) {
    P.lanes.push_back(lane);
    lane = HostLane{};
    return;
  }
  lk.unlock();
  free_lane(lane);
}

hipError_t DevPack::commit(DevBuf<char>& arena, hipStream_t s) {
  size_t total = 0;
  for (const Item& i : items_)
    if (i.size * i.count <= kPackBytes) total += (i.size * i.count + kAlign - 1) / kAlign * kAlign;
  std::vector<char> host(total, 0);
  hipError_t e = arena.alloc(total);
  size_t at = 0;
  for (const Item& i : items_) {
    if (e != hipSuccess) return e;
    const size_t bytes = i.size * i.count;
    if (bytes == 0) continue;
    if (bytes <= kPackBytes) {
      e = i.place(i.buf, arena.p + at, i.count);
      if (i.data) std::memcpy(host.data() + at, i.data, bytes);
      at += (bytes + kAlign - 1) / kAlign * kAlign;
      continue;
    }
    e = i.place(i.buf, nullptr, i.count);
    if (e != hipSuccess) return e;
    e = i.data ? copy_now(i.where(i.buf), i.data, bytes, hipMemcpyHostToDevice, s)
               : hipMemsetAsync(i.where(i.buf), 0, bytes, s);
  }
  items_.clear();
  if (e != hipSuccess || total == 0) return e;
  return copy_now(arena.p, host.data(), total, hipMemcpyHostToDevice, s);
}

void transfer_open() {
  Pool& P = pool();
  std::lock_guard<std::mutex> lk(P.mu);
  P.users += 1;
}

void transfer_close() {
  std::vector<Slot> drop;
  std::vector<HostLane> lanes;
  {
    Pool& P = pool();
    std::lock_guard<std::mutex> lk(P.mu);
    if (--P.users == 0) {
      drop.swap(P.idle);
      lanes.swap(P.lanes);
    }
  }
  for (Slot& s : drop) free_slot(s);
  for (HostLane& l : lanes) free_lane(l);
}

int export_sites(hlb_lattice* h, const TransferPart* parts, int count, bool shifted) {
  const int64_t N = h->L.N;
  TransferPart used[kMaxTransferParts];
  int np = 0;
  int64_t row = 0, widest = 0;  // doubles per site, of all parts and of the largest
  for (int i = 0; i < count; ++i)
    if (parts[i].host) {
      used[np++] = parts[i];
      row += parts[i].planes;
      widest = std::max<int64_t>(widest, parts[i].planes);
    }
  if (N == 0 || np == 0) {
    HLB_CHECK(hipStreamSynchronize(h->stream));
    return HLB_OK;
  }
  const int64_t per = (int64_t)(kSlotBytes / sizeof(double)) / row / 64 * 64;
  const int64_t chunks = (N + per - 1) / per;
  auto start = [&](char* slot, int64_t c) -> int {
    Chunk a{};
    const int64_t k0 = c * per, n = std::min<int64_t>(per, N - k0);
    int64_t at = 0;
    for (int i = 0; i < np; ++i) {
      a.part[i] = ChunkPart{used[i].device, used[i].planes, (int32_t)at};
      at += n * used[i].planes;
    }
    a.slot = h->dinv.p + k0;
    a.S = h->S;
    a.n = (int32_t)n;
    const dim3 grid(blocks_for(n * widest), (unsigned)np);
    double* out = reinterpret_cast<double*>(slot);
    if (shifted) hipLaunchKernelGGL(export_chunk<float>, grid, dim3(kBlock), 0, h->stream, a, out);
    else hipLaunchKernelGGL(export_chunk<double>, grid, dim3(kBlock), 0, h->stream, a, out);
    HLB_CHECK(hipGetLastError());
    return HLB_OK;
  };
  auto finish = [&](const char* slot, int64_t c) {
    const int64_t k0 = c * per, n = std::min<int64_t>(per, N - k0);
    const double* from = reinterpret_cast<const double*>(slot);
    for (int i = 0; i < np; ++i) {
      const int64_t w = used[i].planes;
      std::memcpy(used[i].host + k0 * w, from, sizeof(double) * (size_t)(n * w));
      from += n * w;
    }
  };
  return run_chunks(h, chunks, sizeof(double) * (size_t)(N * row), start, finish);
}

int import_sites(hlb_lattice* h, const double* f, void* planes, bool shifted) {
  const int64_t N = h->L.N;
  if (N == 0) return HLB_OK;
  const int64_t per = (int64_t)(kSlotBytes / sizeof(double)) / Q / 64 * 64;
  const int64_t chunks = (N + per - 1) / per;
  auto start = [&](char* slot, int64_t c) -> int {
    const int64_t k0 = c * per, n = std::min<int64_t>(per, N - k0);
    std::memcpy(slot, f + k0 * Q, sizeof(double) * (size_t)(n * Q));
    const dim3 grid(blocks_for(n * Q));
    const double* in = reinterpret_cast<const double*>(slot);
    if (shifted)
      hipLaunchKernelGGL(import_chunk<float>, grid, dim3(kBlock), 0, h->stream, in, h->dinv.p + k0, (int32_t)n, h->S,
                         static_cast<float*>(planes));
    else
      hipLaunchKernelGGL(import_chunk<double>, grid, dim3(kBlock), 0, h->stream, in, h->dinv.p + k0, (int32_t)n, h->S,
                         static_cast<double*>(planes));
    HLB_CHECK(hipGetLastError());
    return HLB_OK;
  };
  return run_chunks(h, chunks, sizeof(double) * (size_t)(N * Q), start, [](const char*, int64_t) {});
}

}  // namespace hlb
