// windkessel.h -- the Windkessel iolets' share of a step launch.
//
// InOutLetWK*::DoComms (InOutLetWK3.cc:33-52) of step t scales the flux sum of
// step t - 1, and the pressure update of step t (InOutLetWK2.cc:82-95,
// InOutLetWK3.cc:70-95) uses that scaled flow: the ghost density of step t + 1
// depends on the sum of step t - 1, not of step t.  So the first workgroups of
// step t's own launch, one per Windkessel iolet, sum what step t - 1 left and
// form the density of step t + 1 while the rest of the launch advances the
// lattice; the coupling terms alternate between two buffers.  A sequence of
// steps starts with the first row's densities (wk_start) and ends with the
// last step's sum (wk_flush), which leaves the state the reference has between
// steps.
//
// Before, each step ran two more launches in line, one that formed the
// densities and one that summed (4.9 and 17.5 us on the 3M-site FP64 tree with
// 8 outlets).  Steps of that tree 214 -> 201 us, of the 7.6M-site FP32 tree with
// 16 outlets 255 -> 251 us.
//
// FP64 form: the terms are added in the reference's site order
// (InOutLetWK3.cc:33-52 accumulates flowRateNew += u.(-n) site by site), one
// wavefront reading 64 at a time a chunk ahead of its chain of dependent
// additions, about 7 ns a term.  FP32-shifted form: no order, so 256 strided
// partial sums of four each, combined across lanes in a fixed order, in FP64.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/hemepure_amd.h"
#include "d3q19.h"
#include "device_util.h"
#include "lbm_kernels.h"

namespace hlb {

__device__ __forceinline__ double lane_value(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)b, lane);
  const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(b >> 32), lane);
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}

// 0 + t[0] + t[1] + ... + t[n - 1], in that order, by one wavefront.
__device__ __forceinline__ double chain_sum(const double* t, int n) {
  const int lane = threadIdx.x & 63;
  double sum = 0.0;
  double next = lane < n ? ldp(t, (uint32_t)lane) : 0.0;
  for (int i = 0; i < n; i += 64) {
    const double v = next;
    if (i + 64 + lane < n) next = ldp(t, (uint32_t)(i + 64 + lane));
    if (n - i >= 64) {
#pragma unroll
      for (int k = 0; k < 64; ++k) sum += lane_value(v, k);
    } else {
      for (int k = 0; k < n - i; ++k) sum += lane_value(v, k);
    }
  }
  return sum;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The sum of t[0 .. n - 1] by one wavefront, as four wavefronts of strided
// shares would form it.
__device__ __forceinline__ double tree_sum(const double* t, int n) {
  constexpr int T = 256;
  double part[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
    int e = 64 * w + (int)(threadIdx.x & 63);
    for (; e + 3 * T < n; e += 4 * T) {
      p0 += ldp(t, (uint32_t)e);
      p1 += ldp(t, (uint32_t)(e + T));
      p2 += ldp(t, (uint32_t)(e + 2 * T));
      p3 += ldp(t, (uint32_t)(e + 3 * T));
    }
    for (; e < n; e += T) p0 += ldp(t, (uint32_t)e);
    part[w] = wave_sum((p0 + p1) + (p2 + p3));
  }
  return 0.0 + ((part[0] + part[1]) + (part[2] + part[3]));
}

// Sum of the flux terms step `step` of the sequence left, by one wavefront.
__device__ __forceinline__ double wk_flux_sum(const WkRef& ref, int step) {
  const int32_t lb = __builtin_amdgcn_readfirstlane(ref.w->list_begin);
  const int32_t n = __builtin_amdgcn_readfirstlane(ref.w->list_end) - lb;
  const double* t = ref.contrib + (int64_t)(step & 1) * ref.stride + lb;
  return ref.ordered ? chain_sum(t, n) : tree_sum(t, n);
}

// DoComms, the centre site's pressure update and the post-stream commit
// (InOutLetWK3.cc:97-106) of step `step` of a sequence, and the ghost density
// of the step after it.  One wavefront.
__device__ __forceinline__ void wk_advance(const WkRef& ref, int step, bool last) {
  WkIolet& w = *ref.w;
  double sum = w.flowRateNew, count = w.siteCount;
  if (step > 0) {
    sum = wk_flux_sum(ref, step - 1);
    count = (double)(w.list_end - w.list_begin);
  }
  if ((threadIdx.x & 63) != 0) return;
  const double density = w.densityNew;
  double flow = sum;
  if (count != 0) flow = flow * w.area / count;
  double next = density;
  if (w.centre_coupled) {
    const double pressure = density * CS2;
    if (w.kind == HLB_IOLET_WK2) {
      const double R0 = w.resistance, C0 = w.capacitance;
      const double pressureNew = R0 / (1.0 + R0 * C0) * (flow + C0 * pressure);
      next = pressureNew / CS2;
    } else {
      const double Rc = w.r_c, Rp = w.r_p, Cp = w.capacitance;
      const double pressureNew = (Rp * Cp * pressure + (Rc + Rp) * (2.0 * flow - w.flowRateOld) +
                                  Rc * Rp * Cp * (flow - w.flowRateOld)) /
                                 (1.0 + Rp * Cp);
      next = pressureNew / CS2;
    }
    w.flowRateOld = flow;
  }
  w.density = next;
  w.densityNew = next;
  w.flowRate = flow;
  w.flowRateNew = 0.0;
  w.siteCount = 0.0;
  if (!last) ref.io_dens[(int64_t)(step + 1) * ref.row + ref.g] = next;
}

// True for the launch's leading workgroups, which serve the Windkessel iolets.
__device__ __forceinline__ bool wk_workgroup(const WkLaunch& wk, int step) {
  if (blockIdx.x >= wk.groups) return false;
  if (blockIdx.x < (uint32_t)wk.n && threadIdx.x < 64) wk_advance(wk.refs[blockIdx.x], step, step + 1 == wk.steps);
  return true;
}

}  // namespace hlb
