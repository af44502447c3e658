// Deterministic reductions to the host in one launch: every work-group
// reduces its share, the last one to finish (a ticket counter) combines the
// partial results in their fixed order and writes the result to pinned memory.
#pragma once
#include "gmod_common.h"

namespace gmod {

constexpr int RED_TPB = 256;

// work-groups for n elements: one per 1024, at most RED_MAX_BLOCKS
inline int red_blocks(long n) {
  const long b = (n + 1023) / 1024;
  return (int)(b < 1 ? 1 : b > RED_MAX_BLOCKS ? RED_MAX_BLOCKS : b);
}

struct RedSum {
  static __device__ double id() { return 0.0; }
  static __device__ double op(double a, double b) { return a + b; }
};
struct RedMax {
  static __device__ double id() { return -HUGE_VAL; }
  static __device__ double op(double a, double b) { return fmax(a, b); }
};
struct RedMin {
  static __device__ double id() { return HUGE_VAL; }
  static __device__ double op(double a, double b) { return fmin(a, b); }
};

// v: this thread's values -> on thread 0 the work-group's (RED_TPB threads)
template <class Op, int W>
__device__ __forceinline__ void block_reduce(double (&v)[W], double* sh) {
#pragma unroll
  for (int c = 0; c < W; ++c) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v[c] = Op::op(v[c], __shfl_down(v[c], o));
    if ((threadIdx.x & 63) == 0) sh[c * (RED_TPB / 64) + (threadIdx.x >> 6)] = v[c];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < W; ++c) {
      double r = sh[c * (RED_TPB / 64)];
#pragma unroll
      for (int w = 1; w < RED_TPB / 64; ++w) r = Op::op(r, sh[c * (RED_TPB / 64) + w]);
      v[c] = r;
    }
  }
  __syncthreads();
}

// The launch's result for the nb work-groups b = 0 .. nb - 1: out[0 .. W) and,
// when err is given, out[W] = its value (an error flag read along).  part has
// room for nb W values, *ticket is zero before and after.
template <class Op, int W>
__device__ __forceinline__ void finish_reduce(double (&v)[W], int b, int nb, double* part, unsigned* ticket,
                                              double* out, const int* err = nullptr) {
  __shared__ double sh[W * (RED_TPB / 64)];
  __shared__ unsigned last;
  block_reduce<Op, W>(v, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < W; ++c) part[W * b + c] = v[c];
    __threadfence();
    last = atomicAdd(ticket, 1u) == (unsigned)nb - 1u;
  }
  __syncthreads();
  if (!last) return;
  __threadfence();
  double r[W];
#pragma unroll
  for (int c = 0; c < W; ++c) r[c] = Op::id();
  for (int i = threadIdx.x; i < nb; i += RED_TPB) {
#pragma unroll
    for (int c = 0; c < W; ++c)
      r[c] = Op::op(r[c], __hip_atomic_load(part + W * i + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  }
  block_reduce<Op, W>(r, sh);
  if (threadIdx.x == 0) {
#pragma unroll
    for (int c = 0; c < W; ++c) out[c] = r[c];
    if (err) out[W] = (double)*err;
    *ticket = 0u;
  }
}

}  // namespace gmod
