// transfer.h -- reordered copies between device planes (slot order) and host
// site records (the reference's site order).
#pragma once

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

// The device copy of the site -> slot index and the handle's share of the
// pinned chunks; closed once when the handle goes.
int transfer_open(hlb_lattice* h);
void transfer_close();

// Both follow the work queued on the handle's stream and return when the host
// arrays are complete.  shifted: the planes are float g = f - w rather than
// double.
int export_sites(hlb_lattice* h, const TransferPart* parts, int count, bool shifted);
int import_sites(hlb_lattice* h, const double* f, void* planes, bool shifted);

}  // namespace hlb
