// transfer.h -- reordered copies between device planes (slot order) and host
// site records (the reference's site order).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

struct hlb_lattice;

namespace hlb {

constexpr int kMaxTransferParts = 6;

// `planes` (1, 3, 6, 17 or 19) device planes of stride S to `host`: planes
// doubles per site; a null host array is skipped.
struct TransferPart {
  const void* device;
  int32_t planes;
  double* host;
};

// A stream with two timing events and pinned staging, which a lattice has from
// its first use to its end.  Making one costs ~0.6 ms and dropping it ~0.4 ms,
// so idle ones are kept (up to kIdleLanes, none once no user is left).
struct HostLane {
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double* stage = nullptr;  // pinned
  size_t doubles = 0;
  int device = -1;
};
int take_lane(int device, size_t doubles, HostLane& out);
void give_lane(HostLane& lane);  // the stream is idle

// A user of the pinned chunks and lanes (a lattice with a device state, a
// server, whose lattices come and go); closed once when it goes.
void transfer_open();
void transfer_close();

// Both follow the work queued on the handle's stream and return when the host
// arrays are complete.  shifted: the planes are float g = f - w rather than
// double.
int export_sites(hlb_lattice* h, const TransferPart* parts, int count, bool shifted);
int import_sites(hlb_lattice* h, const double* f, void* planes, bool shifted);

}  // namespace hlb
