// Shared definitions for the simkit_amd HIP library (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/simkit_amd.h"

namespace sk {

// Newton's relative-gradient test ||g|| <= rtol ||g(x0)|| cannot be met once
// the accepted update no longer changes the positions: when
// max |t dx| <= kStepFloor max |x| over the free DOFs (4 machine epsilons, the
// spacing of doubles near max |x|), further iterations only re-round x, and
// the iterate is converged to working precision. This only binds when x0 is
// already an equilibrium to within that resolution (a damped mesh at rest),
// where ||g(x0)|| itself is tiny. newton.py:69 stops on the step length too.
constexpr double kStepFloor = 4.0 * 2.220446049250313e-16;

// Whether a material reads lam (every density except ARAP).
constexpr bool material_needs_lam(int material) { return material != SK_ARAP; }

// Last error message of the calling host thread (returned by sk_last_error).
void set_error(const std::string& msg);

#define SK_HIP_CHECK(expr)                                                            \
  do {                                                                                \
    hipError_t _e = (expr);                                                           \
    if (_e != hipSuccess) {                                                           \
      ::sk::set_error(std::string(#expr) + ": " + hipGetErrorString(_e));             \
      return SK_ERR_HIP;                                                              \
    }                                                                                 \
  } while (0)

#define SK_REQUIRE(cond, msg)                                                         \
  do {                                                                                \
    if (!(cond)) {                                                                    \
      ::sk::set_error(msg);                                                           \
      return SK_ERR_INVALID;                                                          \
    }                                                                                 \
  } while (0)

#define SK_TRY(expr)                                                                  \
  do {                                                                                \
    int _s = (expr);                                                                  \
    if (_s != SK_OK) return _s;                                                       \
  } while (0)

// f(), which returns a status; an exception of the host code (no memory)
// becomes one, since none may leave a C entry point or a host thread.
template <typename F>
int no_throw(F&& f) {
  try {
    return f();
  } catch (...) {
    try {
      set_error("out of host memory");
    } catch (...) {
    }
    return SK_ERR_HIP;
  }
}

constexpr int kWave = 64;
constexpr int kBlock = 256;

inline int grid_for(long long n, int block = kBlock) {
  long long g = (n + block - 1) / block;
  return static_cast<int>(g < 1 ? 1 : g);
}

// ---------------------------------------------------------------------------
// Deterministic reductions. A block reduces in a fixed tree (wave shuffles,
// then LDS across the 4 waves of a 256-thread block); a grid reduction writes
// one partial per block and the last block to finish sums the partials in a
// fixed order, so results are bit-reproducible for a fixed launch shape.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = kWave / 2; off > 0; off >>= 1) v += __shfl_down(v, off, kWave);
  return v;
}

// Sum over the wave in lane 63 (fixed tree of DPP row shifts and broadcasts).
template <int kCtrl, int kRows>
__device__ __forceinline__ double dpp_add(double v) {
  const uint64_t u = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, kCtrl, kRows, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), kCtrl, kRows, 0xf, true);
  return v + __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
template <int kCtrl, int kRows>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, kRows, 0xf, true));
}
template <typename T>
__device__ __forceinline__ T wave_sum_last(T v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8: prefix sums of the rows of 16 lanes
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast 15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast 31 into rows 2 and 3
  return v;
}

// Barrier that orders LDS only: the workgroup's waves share nothing else inside
// the loop, and __syncthreads would also wait for the words just stored.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// x, of unknown value to the compiler: what is computed from it inside the
// iteration (addresses, unpacked fields) is not hoisted out of it into
// registers that the matrix blocks need.
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Orders a wave's LDS accesses among its lanes (the wave's own accesses are in order).
__device__ __forceinline__ void wave_lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// The FP16 values in the low and high halves of a 32-bit word.
__device__ __forceinline__ float half_lo(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w & 0xFFFFu)); }
__device__ __forceinline__ float half_hi(uint32_t w) { return (float)__builtin_bit_cast(_Float16, (uint16_t)(w >> 16)); }

template <int NV>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* lds /* NV * kBlock/kWave */) {
  const int lane = threadIdx.x % kWave;
  const int wid = threadIdx.x / kWave;
  constexpr int nw = kBlock / kWave;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  __syncthreads();
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) lds[k * nw + wid] = v[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
#pragma unroll
      for (int w = 0; w < nw; ++w) s += lds[k * nw + w];
      v[k] = s;
    }
  }
}

// Grid reductions without fences or atomics: every block writes its block
// sum to partials[k * gridDim.x + blockIdx.x] with plain stores; a later
// kernel (ordered after this one on the stream) sums the partials in a fixed
// order, either in a dedicated one-block finalize launch or redundantly in
// every block of the consuming kernel. Results are bit-reproducible for a
// fixed launch shape, and no block waits on another block.
template <int NV>
__device__ __forceinline__ void store_block_partials(double (&v)[NV], double* partials) {
  __shared__ double lds[NV * kBlock / kWave];
  block_sum<NV>(v, lds);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) partials[k * gridDim.x + blockIdx.x] = v[k];
  }
}

// Whole-block sum of n partials per value (value k at partials[k * stride + i]);
// every thread of the block receives the totals.
template <int NV>
__device__ __forceinline__ void sum_partials(const double* __restrict__ partials, int n, int stride,
                                             double (&out)[NV]) {
  __shared__ double lds[NV * kBlock / kWave];
  __shared__ double res[NV];
  double acc[NV];
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += partials[k * stride + i];
    acc[k] = s;
  }
  block_sum<NV>(acc, lds);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) res[k] = acc[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) out[k] = res[k];
}

// One-block launch: result[k] = sum of the n partials of value k.
template <int NV>
__global__ __launch_bounds__(kBlock) void finalize_sum_kernel(const double* __restrict__ partials, int n,
                                                              double* __restrict__ result) {
  double out[NV];
  sum_partials<NV>(partials, n, n, out);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < NV; ++k) result[k] = out[k];
  }
}

}  // namespace sk
