// Wave-level device helpers shared by the plain and the batched kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pysa {

__device__ __forceinline__ int rl(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float rl(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ uint32_t rl(uint32_t v, int lane) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, lane);
}
__device__ __forceinline__ uint64_t rl(uint64_t v, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ double rl(double v, int lane) {
  return __longlong_as_double((long long)rl((uint64_t)__double_as_longlong(v), lane));
}

// Orders LDS accesses of one wave across its lanes (the hardware executes them
// in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Replica exchange of one read by one wave (utils.py:44-58): hot end first,
// slot a = R-1-k against b = a-1 at step k.  The replica that the last pair
// left in slot a is carried along: an exchange moves it on to b, otherwise b's
// occupant becomes the carried one.  Lane k holds pair k's other operands, so a
// step is a few readlanes and no memory.  E, beta, lu, bi: shared or global
// arrays of the read; e_of(r): the energy of replica r.
template <typename T, typename I>
__device__ void exchange_wave(int R, const T* E, const T* beta, const double* lu, I* bi) {
  const int lane = threadIdx.x & 63;
  int carry = (int)bi[R - 1];
  T ec = E[carry];
  for (int k0 = 0; k0 < R - 1; k0 += 64) {
    const int cnt = min(64, R - 1 - k0);
    const int k = k0 + min(lane, cnt - 1);
    const int a = R - 1 - k;
    const int rb_l = (int)bi[a - 1];
    const T eb_l = E[rb_l], db_l = (T)(beta[a] - beta[a - 1]);
    const double lu_l = lu[k];
    int out = 0;
    for (int j = 0; j < cnt; ++j) {
      const T eb = rl(eb_l, j);
      const int rb = rl(rb_l, j);
      const T dd = (T)(ec - eb) * rl(db_l, j);
      const bool x = dd >= 0 || rl(lu_l, j) < (double)dd;
      if (lane == j) out = x ? rb : carry;
      if (!x) {
        carry = rb;
        ec = eb;
      }
    }
    if (lane < cnt) bi[a] = (I)out;
  }
  if (lane == 0) bi[0] = (I)carry;
}

}  // namespace pysa
