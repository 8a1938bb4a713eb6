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
// (InOutLetWK3.cc:33-52 accumulates flowRateNew += u.(-n) site by site) by one
// wavefront, a chain of dependent additions that bounds the step of a wide
// outlet.  A term costs one broadcast within its row of 16 lanes and the
// addition, 5.2 ns; taken from its lane through two scalar registers it cost
// 10.1 ns, from LDS in a launch of its own 7.4 ns.  FP32-shifted form: no order,
// so 256 strided partial sums of four each, combined across lanes in a fixed
// order, in FP64; the one wavefront has all 16 loads of 1024 terms in flight, for
// with four at a time a wide outlet's sum outlasted the step.
//   us a step, outlet of 11,300 sites (0.27M-site pipe) FP64 115.5 -> 59.2,
//   31,400 sites (0.75M) FP64 316 -> 162, FP32 50 -> 27.5; 5,000 sites FP64 56
//   -> 33; 1,260 sites FP64 15.9 -> 8.8.
//
// No intrinsic with a side effect belongs here (raised wave priority): the
// compiler takes it for a write to memory and reads the slab records of every
// wave of the step with vector loads instead of scalar ones (FP32 ensemble 26.8
// -> 31.2 ms a pass, 7.6M-site tree 84 -> 94).
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

// s + v of lane 0 + v of lane 1 + ... + v of lane 15 of each lane's row of 16, in
// that order: one broadcast within the row and one addition a term.
template <int K = 0>
__device__ __forceinline__ double row_chain(double s, double v) {
  if constexpr (K < 16) return row_chain<K + 1>(s + __builtin_amdgcn_mov_dpp(v, 0x150 + K, 0xf, 0xf, true), v);
  else return s;
}

// 0 + t[0] + t[1] + ... + t[n - 1], in that order, by one wavefront: 64 terms a
// load, kChainAhead loads ahead of the additions.
constexpr int kChainAhead = 4;
__device__ __forceinline__ double chain_sum(const double* t, int n) {
  const int lane = threadIdx.x & 63;
  double ahead[kChainAhead];
#pragma unroll
  for (int a = 0; a < kChainAhead; ++a) ahead[a] = 64 * a + lane < n ? ldp(t, (uint32_t)(64 * a + lane)) : 0.0;
  double sum = 0.0;
  int i = 0;
  for (; i + 64 <= n; i += 64) {
    const double v = ahead[0];
#pragma unroll
    for (int a = 1; a < kChainAhead; ++a) ahead[a - 1] = ahead[a];
    const int e = i + 64 * kChainAhead + lane;
    if (e < n) ahead[kChainAhead - 1] = ldp(t, (uint32_t)e);
#pragma unroll
    for (int r = 0; r < 4; ++r) sum = lane_value(row_chain(sum, v), 16 * r);
  }
  int k = 0;
  for (; i + k + 16 <= n; k += 16) sum = lane_value(row_chain(sum, ahead[0]), k);
  for (; i + k < n; ++k) sum += lane_value(ahead[0], k);
  return sum;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// The sum of t[0 .. n - 1] by one wavefront, as four wavefronts of strided
// shares with four partial sums a lane would form it; all 16 loads of a round are
// in flight together.
__device__ __forceinline__ double tree_sum(const double* t, int n) {
  constexpr int T = 256;
  const int lane = threadIdx.x & 63;
  double p[4][4] = {};
  int base = 0;
  for (; base + 4 * T <= n; base += 4 * T) {
    double v[4][4];
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int k = 0; k < 4; ++k) v[w][k] = ldp(t, (uint32_t)(base + k * T + 64 * w + lane));
#pragma unroll
    for (int w = 0; w < 4; ++w)
#pragma unroll
      for (int k = 0; k < 4; ++k) p[w][k] += v[w][k];
  }
  double part[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    int e = base + 64 * w + lane;
    if (e + 3 * T < n) {
#pragma unroll
      for (int k = 0; k < 4; ++k) p[w][k] += ldp(t, (uint32_t)(e + k * T));
      e += 4 * T;
    }
    for (; e < n; e += T) p[w][0] += ldp(t, (uint32_t)e);
    part[w] = wave_sum((p[w][0] + p[w][1]) + (p[w][2] + p[w][3]));
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
