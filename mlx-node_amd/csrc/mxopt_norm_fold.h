// The end of a norm: every workgroup's partial sum, their fold and what follows from it.
#pragma once
#include "mxopt_kernels_common.h"

namespace mxopt {

// Sum of n partial sums by the THREADS lanes of one workgroup, in an order that depends on n and THREADS alone; valid on thread
// 0.  Bound by the latency of memory round trips, not by bytes (16,384 partials are 128 KB): every lane issues its next
// kFoldLoads loads before it adds the first of them.  Microseconds of the second pass with 8 loads and 256 lanes up to 2,048 partial
// sums, and with 16 and 256 up to 4,096 (which adds 2,049 - 4,096 of them in another order): 100 1.7 and 1.9, 2,048 1.9 and 2.0, 2,049 2.3
// and 2.0, 4,096 3.8 and 2.2, 8,192 4.4 and 3.9, 16,384 4.6 and 4.6.  SHARED: other workgroups of the same launch have written them.
constexpr int kFoldLoads = 16;
template <int THREADS, bool SHARED>
__device__ __forceinline__ double sum_of_partials(const double* partials, uint32_t n) {
  __shared__ double wave_sums[THREADS / 64];
  const MXOPT_GLOBAL double* part = global_ptr<double>((const void*)partials);
  double s = 0.0;
  for (uint32_t base = 0; base < n; base += THREADS * kFoldLoads) {
    double x[kFoldLoads];
#pragma unroll
    for (int k = 0; k < kFoldLoads; ++k) {
      const uint32_t i = base + (uint32_t)k * THREADS + threadIdx.x;
      if (SHARED) x[k] = i < n ? __hip_atomic_load(part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0.0;
      else x[k] = i < n ? part[i] : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kFoldLoads; ++k) s += x[k];
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63u) == 0) wave_sums[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    s = wave_sums[0];
#pragma unroll
    for (int w = 1; w < THREADS / 64; ++w) s += wave_sums[w];
  }
  return s;
}

__device__ __forceinline__ mxopt_norm_result norm_outcome(double sumsq, double max_norm, int has_max, int clip_mode) {
  const double norm = sqrt(sumsq);
  const float norm32 = (float)norm;
  float scale = 1.0f;
  if (has_max) {
    if (clip_mode == MXOPT_CLIP_ALWAYS_MULTIPLY) {
      // optimizers/mod.rs:87-96: all float32 scalars
      float d = norm32 + (float)1e-6;
      float q = (float)max_norm / d;
      scale = (q != q) ? q : fminf(q, 1.0f);  // a NaN norm gives a NaN scale
    } else {
      // gradients/mod.rs:255-270: float64 on the host, gradients unchanged when norm <= max
      if (!(norm <= max_norm)) scale = (float)(max_norm / (norm + 1e-6));
    }
  }
  mxopt_norm_result r;
  r.sumsq = sumsq;
  r.norm = norm;
  r.norm_f32 = norm32;
  r.scale = scale;
  // NaN: some element was a NaN or an infinity (1).  +Inf: every element was finite and their squares left
  // float32 range (2): the reference goes on with a clip factor of 0 there, and so does `scale` above.
  r.nonfinite = (sumsq != sumsq) ? 1ull : (sumsq - sumsq == 0.0) ? 0ull : 2ull;
  return r;
}

__device__ __forceinline__ void write_outcome(double sumsq, const NormFold& fold) {
  const mxopt_norm_result r = norm_outcome(sumsq, fold.max_norm, fold.has_max, fold.clip_mode);
  *fold.out = r;
  if (fold.host_out != nullptr) {
    *fold.host_out = r;
    __threadfence_system();
  }
}

// The lanes' float64 sums become the workgroup's partial sum; the workgroup that stores the last one of the call folds them
// all, where they are at most kMaxFolded.  The count is never reset: every call knows which arrival is its last one, so that
// calls that should have been ordered and were not leave nothing behind for the next.  It saves a launch, not device time.  Global norm, microseconds a call with a second
// kernel and with the fold, called from a loop: 1,000 elements (1 partial sum) 7.4 and 4.4, 60 chunks 8.0 and 6.0; replayed from a
// graph 12 chunks 4.5 and 4.5, 60 4.6 and 4.9.  With 1,024 partial sums and their arrivals counted in two stages the
// device takes 5.5 and 5.9, in one stage (an arrival every 12 ns at one counter) 16.
__device__ __forceinline__ void finish_partial(double acc_sum, double* __restrict__ partial_sum, const NormFold& fold) {
  unsigned long long unused = 0;
  block_sum(acc_sum, unused);
  if (fold.count == 0) {
    if (threadIdx.x == 0) partial_sum[blockIdx.x] = acc_sum;
    return;
  }
  __shared__ uint32_t last;
  if (threadIdx.x == 0) {
    // Written through to where every compute die sees it, and arrived there, before the arrival is counted.  (A release fence
    // would also write the die's whole L2 back.)
    __hip_atomic_store(partial_sum + blockIdx.x, acc_sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    last = __hip_atomic_fetch_add(fold.arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == fold.last_arrival;
  }
  __syncthreads();
  if (!last) return;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
  const double s = sum_of_partials<kThreads, true>(fold.partials, fold.count);
  if (threadIdx.x == 0) write_outcome(s, fold);
}

}  // namespace mxopt
