// Device code shared by the kernel translation units: the reference's op chains as math functors,
// the chunk lookup, the norm's per-element value and the launch macro.
#pragma once

#include "mxopt_device.h"
#include "mxopt_launch.h"

namespace mxopt {

// ------------------------------------------------------------------------------------
// Math functors: the reference's op chains, one rounded float32 operation per line.
// ------------------------------------------------------------------------------------

// mlx square is a unary op and keeps its operand's dtype (mlx.cpp:2016-2020): the square of a 16-bit
// gradient that reaches it as it came (no prep stage, no pending sum, no coupled decay in front of it)
// is a 16-bit tensor, and only the multiply by the float32 scalar that follows promotes it.  g * g is
// exact in float32 for 16-bit inputs, so rounding it once is that tensor.
__device__ __forceinline__ float round_square_to(int dtype, float sq) {
  if (dtype == MXOPT_BF16) return Elem<MXOPT_BF16>::round(sq);
  if (dtype == MXOPT_F16) return Elem<MXOPT_F16>::round(sq);
  return sq;
}

// Adam::update_single (optimizers/adam.rs:77-108) / AdamW::update_single (adamw.rs:81-116).
struct AdamMath {
  mxopt_adam_hp hp;
  int gsq_dtype = MXOPT_F32;  // dtype the square of the gradient is rounded to (adamw.rs:92, adam.rs:88)
  static constexpr bool kM = true, kV = true, kSquare = true;
  __device__ __forceinline__ bool uses_v(uint32_t) const { return true; }
  __device__ __forceinline__ bool reads_v(uint32_t) const { return true; }
  __device__ __forceinline__ bool rounds_square() const { return gsq_dtype != MXOPT_F32; }
  __device__ __forceinline__ float squared(float, float g) const { return g; }
  __device__ __forceinline__ void operator()(float& p, float g, float& m, float& v, float bc1, float bc2,
                                             uint32_t flags) const {
    apply(p, g, m, v, bc1, bc2, flags, round_square_to(gsq_dtype, g * g));
  }
  // gsq: the square of squared(p, g), rounded to gsq_dtype.
  __device__ __forceinline__ void apply(float& p, float g, float& m, float& v, float bc1, float bc2, uint32_t,
                                        float gsq) const {
    float pd = hp.decoupled_decay ? p * hp.decay : p;
    float b1m = m * hp.beta1;
    float g1 = g * hp.one_minus_beta1;
    float nm = b1m + g1;
    float b2v = v * hp.beta2;
    float g2 = gsq * hp.one_minus_beta2;
    float nv = b2v + g2;
    float mh = nm * bc1;  // bc == 1.0f reproduces "bias correction off" exactly
    float vh = nv * bc2;
    float den = sqrtf(vh) + hp.eps;
    float u = mh / den;
    float lu = u * hp.lr;
    p = pd - lu;
    m = nm;
    v = nv;
  }
};

// SGD::update_single (optimizers/sgd.rs:84-150).
struct SgdMath {
  mxopt_sgd_hp hp;
  static constexpr bool kM = false, kV = true, kSquare = false;
  __device__ __forceinline__ bool uses_v(uint32_t) const { return hp.has_momentum != 0; }
  __device__ __forceinline__ bool reads_v(uint32_t flags) const { return hp.has_momentum && !(flags & kTfFirst); }
  __device__ __forceinline__ bool rounds_square() const { return false; }
  __device__ __forceinline__ void operator()(float& p, float g, float& m, float& v, float bc1, float bc2,
                                             uint32_t flags) const {
    apply(p, g, m, v, bc1, bc2, flags, 0.0f);
  }
  __device__ __forceinline__ void apply(float& p, float g, float&, float& v, float, float, uint32_t flags, float) const {
    float ge = g;
    if (hp.has_weight_decay) {
      float w = p * hp.weight_decay;
      ge = g + w;
    }
    float u = ge;
    if (hp.has_momentum) {
      float nv;
      if (flags & kTfFirst) {
        nv = ge * 1.0f;
      } else {
        float mv = v * hp.momentum;
        float dg = ge * hp.one_minus_dampening;
        nv = mv + dg;
      }
      u = hp.nesterov ? nv + ge : nv;
      v = u;
    }
    float lu = u * hp.lr;
    p = p - lu;
  }
};

// RMSprop::update_single (optimizers/rmsprop.rs:67-112).
struct RmspropMath {
  mxopt_rmsprop_hp hp;
  int gsq_dtype = MXOPT_F32;  // as in AdamMath (rmsprop.rs:80)
  static constexpr bool kM = false, kV = true, kSquare = true;
  __device__ __forceinline__ bool uses_v(uint32_t) const { return true; }
  __device__ __forceinline__ bool reads_v(uint32_t) const { return true; }
  __device__ __forceinline__ bool rounds_square() const { return gsq_dtype != MXOPT_F32; }
  __device__ __forceinline__ float squared(float p, float g) const {
    float ge = g;
    if (hp.has_weight_decay) {
      float w = p * hp.weight_decay;
      ge = g + w;
    }
    return ge;
  }
  __device__ __forceinline__ void operator()(float& p, float g, float& m, float& v, float bc1, float bc2,
                                             uint32_t flags) const {
    const float ge = squared(p, g);
    apply(p, g, m, v, bc1, bc2, flags, round_square_to(gsq_dtype, ge * ge));
  }
  __device__ __forceinline__ void apply(float& p, float g, float&, float& v, float, float, uint32_t, float gsq) const {
    const float ge = squared(p, g);
    float av = v * hp.alpha;
    float g2 = gsq * hp.one_minus_alpha;
    float nv = av + g2;
    float den = sqrtf(nv) + hp.eps;
    float u = ge / den;
    float lu = u * hp.lr;
    p = p - lu;
    v = nv;
  }
};

// Qwen3Model::apply_gradients (models/qwen3/model.rs:2434-2451): lr already rounded to the
// parameter dtype on the host; ROUND_PRODUCT when p and g share a 16-bit dtype (the product
// is then itself a tensor of that dtype).
template <int PD, bool ROUND_PRODUCT>
struct PlainSgdMath {
  float lr_p, weight_decay;
  int has_weight_decay;
  static constexpr bool kM = false, kV = false, kSquare = false;
  __device__ __forceinline__ bool uses_v(uint32_t) const { return false; }
  __device__ __forceinline__ bool reads_v(uint32_t) const { return false; }
  __device__ __forceinline__ bool rounds_square() const { return false; }
  __device__ __forceinline__ void operator()(float& p, float g, float& m, float& v, float bc1, float bc2,
                                             uint32_t flags) const {
    apply(p, g, m, v, bc1, bc2, flags, 0.0f);
  }
  __device__ __forceinline__ void apply(float& p, float g, float&, float&, float, float, uint32_t, float) const {
    float ge = g;
    if (has_weight_decay) {  // sft/engine.rs:345-365: g + f32(wd)*p, promoted to float32
      float w = p * weight_decay;
      ge = g + w;
    }
    float s = lr_p * ge;
    if (ROUND_PRODUCT) s = Elem<PD>::round(s);
    p = p - s;
  }
};

// ------------------------------------------------------------------------------------
// Chunk lookup shared by all kernels
// ------------------------------------------------------------------------------------

struct ChunkView {
  DevTensor t;
  uint64_t start;  // first element of the chunk inside the tensor
  uint32_t len;    // elements in this chunk (kChunk except for the last one)
  uint32_t head;   // chunk 0 of a shifted tensor: elements [0, head) are this workgroup's too
  uint32_t tensor; // row of the table (0 for a single tensor passed by value)
  bool fast;       // full chunk: fully unrolled
};

__device__ __forceinline__ ChunkView locate(const DevTensor* __restrict__ T, const DevChunk* __restrict__ C,
                                            const DevTensor& one, uint32_t c) {
  ChunkView cv;
  uint32_t index;
  if (C != nullptr) {  // table walk: two dependent scalar loads
    const DevChunk ch = load_constant<DevChunk>(C, c);
    cv.t = load_constant<DevTensor>(T, ch.tensor);
    cv.tensor = ch.tensor;
    index = ch.index;
  } else {             // a single tensor described in the kernel arguments: chunk c of `one`
    cv.t = one;
    cv.tensor = 0;
    index = c;
  }
  // The same for the whole workgroup, so it stays in scalar registers: the builder has cut `head` to n, and the number
  // of full chunks fits 32 bits (its limit on n), which leaves no 64-bit compare (there is no scalar one).  Chunks of
  // 10,000 tensors of 2,461 elements: AdamW over four micro-batches 161 -> 143 us, its norm 62 -> 53.
  static_assert(kChunk == 4096, "shift and mask below");
  const uint64_t body = cv.t.n - cv.t.head;
  const uint32_t full = (uint32_t)(body >> 12);
  cv.start = (uint64_t)cv.t.head + (uint64_t)index * kChunk;
  cv.fast = index < full;
  cv.len = cv.fast ? (uint32_t)kChunk : index == full ? (uint32_t)body & (uint32_t)(kChunk - 1) : 0u;
  cv.head = index == 0 ? cv.t.head : 0u;
  return cv;
}

// The engines skip the whole step when any gradient element is NaN/Inf (grpo/engine.rs:561-607):
// with a counter from the norm pass the update kernels honour that without a host round trip.
// Bit 0 of mxopt_norm_result.nonfinite is "some element was a NaN or an infinity"; bit 1 (finite elements
// whose squares overflowed) does not stop a step: the reference clips such gradients to zero and goes on.
__device__ __forceinline__ bool skip_requested(const DevPrep& prep) {
  return prep.d_skip_if_nonzero != nullptr && (*constant_ptr<unsigned long long>(prep.d_skip_if_nonzero) & 1ull) != 0ull;
}

// A value clamp would turn +-Inf into a finite bound and hide it from the sum-based validity
// check; the engines test the raw values (grpo/engine.rs:563-569), so such a lane poisons its partial.

// The value whose square enters the norm.  Under a clamp the lane only has to remember that it met
// a NaN or an infinity (its partial is poisoned afterwards), so the clamp itself can be a single
// median-of-three that does not care about NaN.
__device__ __forceinline__ float norm_value(const PrepRegs& pr, float x, bool clamped, bool& bad) {
  bad |= !__builtin_isfinite(x);
  if (!clamped) return prep_pre(pr, x);
  if (pr.flags & kPrepPreMul) x = x * pr.pre_mul;
  return __builtin_amdgcn_fmed3f(x, pr.pre_lo, pr.pre_hi);
}

// How many workgroups of a launch share a compute unit.  The passes that read and write long lists run at 5.3 - 5.7 TB/s in memory
// of one region with as many as the registers allow, and at 6.1 - 6.5 with fewer, as many as keep some 64 - 100 KB of reads a unit in
// flight: what is in flight, and what is written behind it, then lies in fewer places at a time, and the memory turns from
// reading to writing less often.  Too few leave it waiting; each launcher says what it measured.
struct Crowd {
  int per_cu;         // workgroups (of kThreads) per compute unit
  int fill;           // only where the chunks are at least this full on average, per mille (short chunks need company), and
  int chunks_per_cu;  // only where the launch has at least this many for each compute unit
  // The same in memory that alternates between regions, where there is less to gain.
  int spread_fill, spread_chunks_per_cu;
  constexpr Crowd(int n, int f, int c, int sf, int sc) : per_cu(n), fill(f), chunks_per_cu(c), spread_fill(sf), spread_chunks_per_cu(sc) {}
  constexpr Crowd(int n, int f, int c) : Crowd(n, f, c, f, c) {}
};
constexpr Crowd kNoLimit{0, 0, 0};
constexpr int kNever = 1001;  // per mille

// Dynamic LDS that leaves room for crowd.per_cu workgroups: an equal part of a compute unit's 160 KB in units of its allocation
// (1,280 bytes), one unit less for what a kernel declares itself.
inline uint32_t crowd_lds(const Launch& L, Crowd crowd) {
  const int fill = L.spread ? crowd.spread_fill : crowd.fill, chunks = L.spread ? crowd.spread_chunks_per_cu : crowd.chunks_per_cu;
  if (crowd.per_cu == 0 || (uint64_t)L.nchunks < (uint64_t)chunks * L.num_cus ||
      L.elems * 1000u < (uint64_t)L.nchunks * kChunk * (uint32_t)fill)
    return 0;
  return ((163840u / (uint32_t)crowd.per_cu) / 1280u - 1u) * 1280u;
}

// What a launch was, for mxopt_get_option; hands the LDS on.
inline uint32_t note_launch(const Launch& L, uint32_t lanes, uint32_t workgroups, uint32_t lds) {
  if (L.note != nullptr) *L.note = LaunchNote{lanes, workgroups, lds, 0u};
  return lds;
}

#define MXOPT_LAUNCH_LDS(kernel, lds, L, ...)                                                                            \
  hipLaunchKernelGGL(kernel, dim3((L).grid), dim3(kThreads), note_launch(L, kThreads, (L).grid, lds), (L).stream,      \
                     (L).tensors, (L).chunks, (L).one, (L).nchunks, __VA_ARGS__)
#define MXOPT_LAUNCH_CROWD(kernel, crowd, L, ...) MXOPT_LAUNCH_LDS(kernel, crowd_lds(L, crowd), L, __VA_ARGS__)
#define MXOPT_LAUNCH(kernel, L, ...) MXOPT_LAUNCH_LDS(kernel, 0, L, __VA_ARGS__)

}  // namespace mxopt
