// reduce.hpp -- deterministic wave and block reductions for gfx950.  The tree
// shapes are fixed, so results are reproducible run to run; sums over a grid
// are partials that a later kernel re-sums in a fixed order (kernels.hpp).
#pragma once

#include <hip/hip_runtime.h>

namespace mpp {

constexpr int kWave = 64;

// Wave sum through DPP lane moves instead of LDS-routed shuffles (about 3x
// less latency).  The sequence: quad_perm [1,0,3,2] and [2,3,0,1], row_ror 4
// and 8 (every lane holds its 16-lane row sum), row_bcast 15 and 31 (lane 63
// accumulates the four rows); lane 63's value is then read into every lane.
// Lanes without a DPP source add 0 (update_dpp with old = 0).
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double wave_sum_dpp(double v) {
  v += dpp_move<0xb1>(v);
  v += dpp_move<0x4e>(v);
  v += dpp_move<0x124>(v);
  v += dpp_move<0x128>(v);
  v += dpp_move<0x142>(v);
  v += dpp_move<0x143>(v);
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), 63);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), 63);
  return __hiloint2double(hi, lo);
}

// the same DPP sequence for a float (one 32-bit move per step)
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

__device__ __forceinline__ float wave_sum_dpp(float v) {
  v += dpp_move<0xb1>(v);
  v += dpp_move<0x4e>(v);
  v += dpp_move<0x124>(v);
  v += dpp_move<0x128>(v);
  v += dpp_move<0x142>(v);
  v += dpp_move<0x143>(v);
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// The butterfly sum v += v of lane ^ 32, 16, 8, 4, 2, 1 (every lane holds the
// total), as register moves: permlane32_swap and permlane16_swap pair the
// halves and the rows, row_ror 8 is lane ^ 8, row_ror 4 is lane ^ 4 once the
// values repeat every 8 lanes, quad_perm does lane ^ 2 and ^ 1.  The same
// additions as with shuffles through LDS, bit for bit, without their 12
// round trips of about 100 cycles (6 for a float).
__device__ __forceinline__ void pair_sum32(unsigned v, unsigned &a, unsigned &b, bool rows) {
  const auto r = rows ? __builtin_amdgcn_permlane16_swap(v, v, false, false)
                      : __builtin_amdgcn_permlane32_swap(v, v, false, false);
  a = r[0];
  b = r[1];
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma clang fp contract(off)
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    unsigned l0, l1, h0, h1;
    pair_sum32((unsigned)__double2loint(v), l0, l1, s == 1);
    pair_sum32((unsigned)__double2hiint(v), h0, h1, s == 1);
    v = __hiloint2double((int)h0, (int)l0) + __hiloint2double((int)h1, (int)l1);
  }
  v += dpp_move<0x128>(v);
  v += dpp_move<0x124>(v);
  v += dpp_move<0x4e>(v);
  v += dpp_move<0xb1>(v);
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    unsigned a, b;
    pair_sum32((unsigned)__float_as_int(v), a, b, s == 1);
    v = __int_as_float((int)a) + __int_as_float((int)b);
  }
  v += dpp_move<0x128>(v);
  v += dpp_move<0x124>(v);
  v += dpp_move<0x4e>(v);
  v += dpp_move<0xb1>(v);
  return v;
}

// A block barrier for data in LDS alone: __syncthreads also waits for every
// load in flight from global memory, which this leaves running.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Sum NV values over a block of BS threads; the totals are returned to every
// thread.  lds must hold (BS/64)*NV elements.
template <int NV, int BS, typename T>
__device__ __forceinline__ void block_sum(T (&v)[NV], T *lds) {
  const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  lds_barrier();  // lds may still be read by a previous use
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) lds[w * NV + k] = v[k];
  lds_barrier();
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    T s = 0;
    for (int i = 0; i < BS / kWave; ++i) s += lds[i * NV + k];
    v[k] = s;
  }
}

}  // namespace mpp
