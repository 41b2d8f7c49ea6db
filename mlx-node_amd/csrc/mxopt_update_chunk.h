// One chunk of the optimizer update, shared by the kernels that walk chunk by chunk (mxopt_kernels.hip) and tile by
// tile (mxopt_update_tile.h).
#pragma once
#include "mxopt_kernels_common.h"

namespace mxopt {

// The gradient the update sees: prep(g), prep(g + g2) (an accumulation buffer plus the micro-batch
// that was not written back to it), or g + prep(g2) (the buffer holds already-clipped gradients and
// the pending micro-batch still has to be clipped: grpo/engine.rs:636-661).  G2 >= 0: a second gradient stream of that
// dtype in tensor.g_out is added to g first (one float32 add, rounded to the buffer's dtype GD: the last micro-batch
// folded into the update instead of being written back to the accumulation buffer).
template <int GD, int G2>
struct GradientOf {
  static constexpr bool kHasG2 = G2 >= 0;
  static constexpr int G2D = kHasG2 ? G2 : MXOPT_F32;
  static constexpr bool kSum16 = kHasG2 && GD != MXOPT_F32;  // the sum is what a 16-bit buffer would have held
  static __device__ __forceinline__ float combine(const PrepRegs& pr, float g, float g2) {
    if (!kHasG2) return prep_all(pr, g);
    if (kSum16) return prep_all(pr, Elem<GD>::round(g + g2));
    return (pr.flags & kPrepPendingOnly) ? g + prep_all(pr, g2) : prep_all(pr, g + g2);
  }
  // g[e] = combine(pr, g[e], g2[e]) without a branch.  kStages false: no stage but the clip factor (pr.flags == 0).
  template <bool kStages>
  static __device__ __forceinline__ void combine_row(const PrepRegs& pr, float (&g)[4], float (&g2)[4]) {
    const bool pending_only = kStages && kHasG2 && !kSum16 && (pr.flags & kPrepPendingOnly);
    float x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = !kHasG2 ? g[e] : pending_only ? g2[e] : g[e] + g2[e];
    if (kSum16) round_group<GD, 4>(x);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x[e] = prep_branchless<kStages>(pr, x[e]);
      g[e] = pending_only ? g[e] + x[e] : x[e];
    }
  }
};

// NTP: the parameters' stores stream too, which pays off only where the line was read (p_out == p in every tensor of the
// launch).  A branch on the two pointers here had the compiler merge both stores into plain ones: plain SGD of 596 M bf16 elements
// 674 us, 592 now, of 128 M 146 and 130; bf16 AdamW of 256 M 998 and 951 (with two workgroups per compute unit).
template <int PD, int GD, int OD, int G2, class Math, bool NT, bool NTP>
__device__ __forceinline__ void update_chunk(const ChunkView& cv, uint32_t tid, const Math& math, const PrepRegs& pr) {
  using Gradient = GradientOf<GD, G2>;
  constexpr bool kHasG2 = Gradient::kHasG2, kSum16 = Gradient::kSum16;
  constexpr int G2D = Gradient::G2D;
  // Elements per lane and group.  With a 16-bit stream in the mix, 8 (one 16-byte access of the 16-bit stream,
  // two of every float32 stream) when a second gradient stream is folded in, 4 (8-byte accesses of the 16-bit
  // streams, one 16-byte access of the float32 ones) without: then every access covers whole sectors and can
  // stream (see load_group).  Measured for bf16 AdamW: no difference on a large list (6.05 against 6.07 ms on
  // Qwen3-1.7B), 11 % less time on a list that a few passes of the memory-side cache cover (10,000 small tensors,
  // 2 GB of traffic per step: 0.316 against 0.353 ms) -- accesses that all stream leave a part of the list
  // resident from one step to the next, plain ones push it out.  With the second stream the wider group wins
  // (fewer, larger requests for three 16-bit streams): 8 there.
  constexpr bool kMixed = PD != MXOPT_F32 || GD != MXOPT_F32 || OD != MXOPT_F32 || (kHasG2 && G2D != MXOPT_F32);
  constexpr int E = (kMixed && kHasG2) ? 8 : 4;
  constexpr int U = kElemsPerLane / E;
  auto combine = [&](float g, float g2) { return Gradient::combine(pr, g, g2); };
  const uint64_t start = cv.start;
  const uint32_t len = cv.len, flags = cv.t.flags;
  const float bc1 = cv.t.bc1, bc2 = cv.t.bc2;
  const void* P = cv.t.p;
  void* PO = cv.t.p_out;
  const void* G = cv.t.g;
  const void* G2P = cv.t.g_out;
  float* M = cv.t.m;
  float* V = cv.t.v;
  const bool use_v = math.uses_v(flags), read_v = math.reads_v(flags);
  auto one_element = [&](uint64_t off) {
    float p = Elem<PD>::load(P, off);
    const float ge = combine(Elem<GD>::load(G, off), kHasG2 ? Elem<G2D>::load(G2P, off) : 0.0f);
    float m = Math::kM ? Elem<MXOPT_F32>::load(M, off) : 0.0f;
    float v = read_v ? Elem<MXOPT_F32>::load(V, off) : 0.0f;
    math(p, ge, m, v, bc1, bc2, flags);
    Elem<OD>::store(PO, off, p);
    if (Math::kM) Elem<MXOPT_F32>::store(M, off, m);
    if (use_v) Elem<MXOPT_F32>::store(V, off, v);
  };

  if (cv.fast) {
    // Full chunk: issue every load of the chunk before the first use.
    float p[U][E], g[U][E], g2[U][E], m[U][E], v[U][E];
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint64_t off = start + (uint64_t)(j * kThreads + tid) * E;
      load_group<PD, E, NT>(P, off, p[j]);
      load_group<GD, E, NT>(G, off, g[j]);
      if (kHasG2) load_group<G2D, E, NT>(G2P, off, g2[j]);
      if (Math::kM) load_group<MXOPT_F32, E, NT>(M, off, m[j]);
      if (read_v) load_group<MXOPT_F32, E, NT>(V, off, v[j]);
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
      if (kSum16) {
#pragma unroll
        for (int e = 0; e < E; ++e) g[j][e] = g[j][e] + g2[j][e];
        round_group<GD, E>(g[j]);
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float ge = kSum16 ? prep_all(pr, g[j][e]) : combine(g[j][e], g2[j][e]);
        math(p[j][e], ge, m[j][e], v[j][e], bc1, bc2, flags);
      }
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
      const uint64_t off = start + (uint64_t)(j * kThreads + tid) * E;
      store_group<OD, E, NTP>(PO, off, p[j]);
      if (Math::kM) store_group<MXOPT_F32, E, NT>(M, off, m[j]);
      if (use_v) store_group<MXOPT_F32, E, NT>(V, off, v[j]);
    }
  } else {
    // Last chunk of a tensor.
    const uint32_t ngroups = len / E;
    for (uint32_t q = tid; q < ngroups; q += kThreads) {
      const uint64_t off = start + (uint64_t)q * E;
      float p[E], g[E], g2[E], m[E], v[E];
      load_group<PD, E, false>(P, off, p);
      load_group<GD, E, false>(G, off, g);
      if (kHasG2) load_group<G2D, E, false>(G2P, off, g2);
      if (Math::kM) load_group<MXOPT_F32, E, false>(M, off, m);
      if (read_v) load_group<MXOPT_F32, E, false>(V, off, v);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        math(p[e], combine(g[e], g2[e]), m[e], v[e], bc1, bc2, flags);
      }
      store_group<OD, E, false>(PO, off, p);
      if (Math::kM) store_group<MXOPT_F32, E, false>(M, off, m);
      if (use_v) store_group<MXOPT_F32, E, false>(V, off, v);
    }
    for (uint32_t i = ngroups * E + tid; i < len; i += kThreads) one_element(start + i);
  }
  if (tid < cv.head) one_element(tid);  // elements in front of the first aligned group
}

}  // namespace mxopt
