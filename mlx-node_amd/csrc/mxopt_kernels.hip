// mxopt kernels for gfx950, part 1: the multi-tensor optimizer updates and the gradient transform.
// Every kernel walks a device-side chunk table so that thousands of tensors share one launch; each is
// a pure streaming pass whose roof is HBM bandwidth.  Build with -ffp-contract=off: one IEEE float32
// rounding per reference op.
#include "mxopt_update_tile.h"

namespace mxopt {

// ------------------------------------------------------------------------------------
// Update kernel, chunk by chunk.
// ------------------------------------------------------------------------------------

template <int PD, int GD, int OD, int G2, class Math, bool NT, bool NTP>
__global__ __launch_bounds__(kThreads) void update_kernel(const DevTensor* __restrict__ T,
                                                          const DevChunk* __restrict__ C, DevTensor one,
                                                          uint32_t nchunks, Math math, DevPrep prep) {
  if (skip_requested(prep)) return;
  const PrepRegs pr = load_prep(prep);
  for (uint32_t c = blockIdx.x; c < nchunks; c += gridDim.x)
    update_chunk<PD, GD, OD, G2, Math, NT, NTP>(locate(T, C, one, c), threadIdx.x, math, pr);
}

// ------------------------------------------------------------------------------------
// Gradient transform: g_out = prep(g)
// ------------------------------------------------------------------------------------

// add != 0: g_out = g_out + prep(g) (one float32 add, rounded to g_out's dtype by the store): the
// engines' "clamp, clip-norm, then accumulate" (grpo/engine.rs:636-661) without materialising the
// clipped gradient.
template <int GD, int OD, bool NT, bool ADD>
__global__ __launch_bounds__(kThreads) void transform_kernel(const DevTensor* __restrict__ T,
                                                             const DevChunk* __restrict__ C, DevTensor one,
                                                             uint32_t nchunks, DevPrep prep) {
  constexpr bool add = ADD;
  // Elements per lane and group: 4 when the kernel adds into g_out (every access then covers whole sectors and
  // streams: the GRPO engine's accumulate of clamp * scale, bf16 into float32, 13.0 against 13.4 ms on the
  // Qwen3-8B list) and when it writes float32 (a wavefront's store is one contiguous kilobyte; of 16-bit input in
  // groups of 8 it was every other 16 bytes of two.  bf16, 8 -> 4: 16 M elements 25.1 -> 20.4 us, 63 M 66.4 -> 59.8,
  // 128 M 137.7 -> 133.9, 256 M 267 -> 266, 600 M 620 -> 627, 1.7 G 1,790 -> 1,799; float16 16 M 25.1 -> 20.4, 256 M
  // 272 -> 266, 1.7 G 1,832 -> 1,800), 8 when a 16-bit stream stays 16-bit.
  constexpr int E = (OD != MXOPT_F32 && !ADD) ? 8 : 4;
  constexpr int U = kElemsPerLane / E;
  if (skip_requested(prep)) return;
  const PrepRegs pr = load_prep(prep);
  const uint32_t tid = threadIdx.x;
  for (uint32_t c = blockIdx.x; c < nchunks; c += gridDim.x) {
    const ChunkView cv = locate(T, C, one, c);
    const uint64_t start = cv.start;
    const void* G = cv.t.g;
    void* GO = cv.t.g_out;
    auto one_element = [&](uint64_t off) {
      float t = prep_all(pr, Elem<GD>::load(G, off));
      if (add) t = Elem<OD>::load(GO, off) + t;
      Elem<OD>::store(GO, off, t);
    };
    if (cv.fast) {
      float g[U][E], a[U][E];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const uint64_t off = start + (uint64_t)(j * kThreads + tid) * E;
        load_group<GD, E, NT>(G, off, g[j]);
        if (add) load_group<OD, E, NT>(GO, off, a[j]);
      }
      // The GRPO engine's order -- clamp, then the clip factor -- with its stage flags tested once per
      // chunk: tested per element they cost the 16-bit first pass (6 B/elem) more instruction issue than
      // it has to spare.
      const bool clamp_then_scale =
          (pr.flags & (kPrepPreMul | kPrepClampPre | kPrepClampPost)) == kPrepClampPre && pr.has_scale;
#pragma unroll
      for (int j = 0; j < U; ++j) {
        if (clamp_then_scale) {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            g[j][e] = clamp_median_keep_nan(g[j][e], pr.pre_lo, pr.pre_hi) * pr.scale;
            if (add) g[j][e] = a[j][e] + g[j][e];
          }
        } else {
#pragma unroll
          for (int e = 0; e < E; ++e) {
            g[j][e] = prep_all(pr, g[j][e]);
            if (add) g[j][e] = a[j][e] + g[j][e];
          }
        }
        store_group<OD, E, NT && ADD>(GO, start + (uint64_t)(j * kThreads + tid) * E, g[j]);  // streaming only where the line was read
      }
    } else {
      const uint32_t ngroups = cv.len / E;
      for (uint32_t q = tid; q < ngroups; q += kThreads) {
        float g[E], a[E];
        load_group<GD, E, false>(G, start + (uint64_t)q * E, g);
        if (add) load_group<OD, E, false>(GO, start + (uint64_t)q * E, a);
#pragma unroll
        for (int e = 0; e < E; ++e) {
          g[e] = prep_all(pr, g[e]);
          if (add) g[e] = a[e] + g[e];
        }
        store_group<OD, E, false>(GO, start + (uint64_t)q * E, g);
      }
      for (uint32_t i = ngroups * E + tid; i < cv.len; i += kThreads) one_element(start + i);
    }
    if (tid < cv.head) one_element(tid);
  }
}

// ------------------------------------------------------------------------------------
// Launchers (dtype dispatch)
// ------------------------------------------------------------------------------------

// Microseconds with as many workgroups as the registers allow (4 or 5) and with two: bf16 AdamW, 10,000 tensors of 64 - 65,536
// elements 405 and 367, one of 24 M 93 and 95, 48 M 185 and 181, 96 M 395 and 369; float32, the 10,000 518 and 488; float32 SGD 378 and
// 356.  10,000 tensors of 100 - 3,000 (chunks 27 %
// full) 52 and 86.  Log-uniform lists, per mille full, 16-bit and float32 AdamW, float32 RMSprop: 620 375 and 389, 479 and 450, 328 and
// 363; 681 386 and 381, 491 and 454, 338 and 354; 802 323 and 312, 418 and 377, 286 and 289; 876 368 and 349, 477 and 427, 324 and 318.
// In memory of several regions: 78 M at 802 per mille (93 chunks a unit) bf16 AdamW 280 and 315, RMSprop 253 and 288, the 10,000
// 339 and 356, 306 and 329; 267 M at 933 (273 a unit) 965 and 936, 885 and 857; float32 AdamW and SGD, the 10,000 428 and 417, 309 and
// 299; a micro-batch folded in 96 M 432 and 420.
// 16-bit parameters without the first moment gain nothing (SGD, 32 M: 79 and 86).
template <int PD, int GD, int G2, class Math>
constexpr Crowd update_crowd() {
  constexpr bool kF32 = PD == MXOPT_F32 && GD == MXOPT_F32;
  if (!Math::kM && !(Math::kV && kF32)) return kNoLimit;
  return Crowd{2, 750, 32, 750, Math::kSquare && !(Math::kM && kF32) && G2 < 0 ? 200 : 32};
}
template <int PD, int GD, int G2, class Math>
constexpr Crowd kUpdateCrowd = update_crowd<PD, GD, G2, Math>();

// Whether the stores of parameters that are updated in place stream.  In memory of several regions they do not as long as
// the parameters stay in the 256 MB memory-side cache for whoever reads them next.  Microseconds plain and streaming, the
// same list again and again: bf16 AdamW 48 M 166 and 175, 90 M 307 and 333, 128 M 440 and 476, 160 M 602 and 598; SGD 90 M 191 and
// 211; float32 AdamW 48 M 205 and 221, 72 M 321 and 331, 80 M 375 and 366, RMSprop 72 M 222 and 234; several lists in turn: bf16 AdamW
// 96 M 365 and 357, float32 64 M 315 and 314.  In memory of one region streaming is ahead except for 16-bit parameters of up to 108 MB:
// several lists in turn, mean over 8 - 50 M elements and three places, streaming takes 1.02 times as long for SGD, 1.01 for RMSprop, the
// same for AdamW, on the same list 1.07, 1.05 and 1.04; 56 M AdamW 214 and 221, SGD 137 and 139, float32 SGD 18 M 73 and 65.
// Launches of less than 24 MB of parameters stream, as they may be pieces of a longer list (22 calls over 31 M elements, plain 174.6,
// streaming 171.7), and so do plain SGD and updates with a micro-batch folded in, which gain nothing by plain stores (96 M 105 and 99;
// 48 M 216 and 217).
template <int PD, int G2, class Math>
static bool stream_parameters(const Launch& L) {
  if (!L.in_place) return false;
  if (!Math::kV || G2 >= 0) return true;
  const uint64_t bytes = L.elems * Elem<PD>::kBytes;
  if (bytes < (24ull << 20)) return true;
  return L.spread ? bytes >= (300ull << 20) : PD == MXOPT_F32 || bytes >= (108ull << 20);
}

template <int PD, int GD, int OD, int G2, class Math>
static void launch_update_t(const Launch& L, const Math& math, const DevPrep& prep) {
  if (!L.nontemporal) {
    MXOPT_LAUNCH((update_kernel<PD, GD, OD, G2, Math, false, false>), L, math, prep);
    return;
  }
  if constexpr (OD == PD) {
    if (launch_update_tiles<PD, GD, G2>(L, math, prep)) return;
    if (stream_parameters<PD, G2, Math>(L)) {
      MXOPT_LAUNCH_CROWD((update_kernel<PD, GD, OD, G2, Math, true, true>), (kUpdateCrowd<PD, GD, G2, Math>), L, math, prep);
      if (L.note != nullptr) L.note->streams_parameters = 1;
      return;
    }
  }
  MXOPT_LAUNCH_CROWD((update_kernel<PD, GD, OD, G2, Math, true, false>), (kUpdateCrowd<PD, GD, G2, Math>), L, math, prep);
}

template <int PD, int GD, class Math>
static bool dispatch_od(int od, const Launch& L, const Math& math, const DevPrep& prep) {
  // The output is either float32 (what the reference returns) or the parameter's own dtype.
  if (od == MXOPT_F32) { launch_update_t<PD, GD, MXOPT_F32, -1>(L, math, prep); return true; }
  if (od == PD) { launch_update_t<PD, GD, PD, -1>(L, math, prep); return true; }
  return false;
}

template <int PD, class Math>
static bool dispatch_gd(int gd, int od, const Launch& L, const Math& math, const DevPrep& prep) {
  switch (gd) {
    case MXOPT_F32: return dispatch_od<PD, MXOPT_F32>(od, L, math, prep);
    case MXOPT_BF16: return dispatch_od<PD, MXOPT_BF16>(od, L, math, prep);
    case MXOPT_F16: return dispatch_od<PD, MXOPT_F16>(od, L, math, prep);
  }
  return false;
}

template <class Math>
static bool dispatch_update(int pd, int gd, int od, const Launch& L, const Math& math, const DevPrep& prep) {
  switch (pd) {
    case MXOPT_F32: return dispatch_gd<MXOPT_F32>(gd, od, L, math, prep);
    case MXOPT_BF16: return dispatch_gd<MXOPT_BF16>(gd, od, L, math, prep);
    case MXOPT_F16: return dispatch_gd<MXOPT_F16>(gd, od, L, math, prep);
  }
  return false;
}

// Adam with the last micro-batch folded in: g is the float32 accumulation buffer, g2 any dtype.
template <int PD>
static bool adam_g2_for_pd(int od, int g2d, const Launch& L, const AdamMath& math, const DevPrep& prep) {
  if (od != PD && od != MXOPT_F32) return false;
  const bool same = od == PD;
  switch (g2d) {
    case MXOPT_F32:
      if (same) launch_update_t<PD, MXOPT_F32, PD, MXOPT_F32>(L, math, prep);
      else launch_update_t<PD, MXOPT_F32, MXOPT_F32, MXOPT_F32>(L, math, prep);
      return true;
    case MXOPT_BF16:
      if (same) launch_update_t<PD, MXOPT_F32, PD, MXOPT_BF16>(L, math, prep);
      else launch_update_t<PD, MXOPT_F32, MXOPT_F32, MXOPT_BF16>(L, math, prep);
      return true;
    case MXOPT_F16:
      if (same) launch_update_t<PD, MXOPT_F32, PD, MXOPT_F16>(L, math, prep);
      else launch_update_t<PD, MXOPT_F32, MXOPT_F32, MXOPT_F16>(L, math, prep);
      return true;
  }
  return false;
}

bool launch_adam(int pd, int gd, int od, int g2d, const Launch& L, const mxopt_adam_hp& hp, const DevPrep& prep) {
  if (g2d < 0) return dispatch_update(pd, gd, od, L, AdamMath{hp, prep_promotes(prep) ? MXOPT_F32 : gd}, prep);
  if (gd != MXOPT_F32) return false;
  switch (pd) {
    case MXOPT_F32: return adam_g2_for_pd<MXOPT_F32>(od, g2d, L, AdamMath{hp}, prep);
    case MXOPT_BF16: return adam_g2_for_pd<MXOPT_BF16>(od, g2d, L, AdamMath{hp}, prep);
    case MXOPT_F16: return adam_g2_for_pd<MXOPT_F16>(od, g2d, L, AdamMath{hp}, prep);
  }
  return false;
}
bool launch_sgd(int pd, int gd, int od, const Launch& L, const mxopt_sgd_hp& hp, const DevPrep& prep) {
  return dispatch_update(pd, gd, od, L, SgdMath{hp}, prep);
}
bool launch_rmsprop(int pd, int gd, int od, const Launch& L, const mxopt_rmsprop_hp& hp, const DevPrep& prep) {
  // with coupled decay the square is taken of g + wd * p, already float32 (rmsprop.rs:69-80)
  const int gsq_dtype = (prep_promotes(prep) || hp.has_weight_decay) ? MXOPT_F32 : gd;
  return dispatch_update(pd, gd, od, L, RmspropMath{hp, gsq_dtype}, prep);
}

template <int PD>
static bool plain_for_pd(int gd, int od, const Launch& L, float lr_p, float wd, int has_wd, bool g_promoted,
                         const DevPrep& prep) {
  if (od != PD) return false;  // apply_gradients always hands back the parameter's dtype
  const bool round_product = (PD != MXOPT_F32) && gd == PD && !g_promoted;
  if (round_product) {
    PlainSgdMath<PD, true> m{lr_p, wd, has_wd};
    return dispatch_gd<PD>(gd, od, L, m, prep);
  }
  PlainSgdMath<PD, false> m{lr_p, wd, has_wd};
  return dispatch_gd<PD>(gd, od, L, m, prep);
}

// Plain SGD on (float32 accumulation buffer + prep(pending gradient)), or on prep(16-bit buffer + pending gradient of
// the same dtype); output in the parameter's dtype.
template <int PD>
static bool plain_pending_for_pd(int gd, int g2d, const Launch& L, float lr_p, float wd, int has_wd, const DevPrep& prep) {
  PlainSgdMath<PD, false> m{lr_p, wd, has_wd};
  if (gd == MXOPT_BF16) { launch_update_t<PD, MXOPT_BF16, PD, MXOPT_BF16>(L, m, prep); return true; }
  if (gd == MXOPT_F16) { launch_update_t<PD, MXOPT_F16, PD, MXOPT_F16>(L, m, prep); return true; }
  switch (g2d) {
    case MXOPT_F32: launch_update_t<PD, MXOPT_F32, PD, MXOPT_F32>(L, m, prep); return true;
    case MXOPT_BF16: launch_update_t<PD, MXOPT_F32, PD, MXOPT_BF16>(L, m, prep); return true;
    case MXOPT_F16: launch_update_t<PD, MXOPT_F32, PD, MXOPT_F16>(L, m, prep); return true;
  }
  return false;
}

bool launch_sgd_plain_pending(int pd, int gd, int od, int g2d, const Launch& L, float lr_p, float wd, int has_wd,
                              const DevPrep& prep) {
  if (od != pd) return false;
  if (gd != MXOPT_F32 && (gd != g2d || (prep.flags & kPrepPendingOnly))) return false;
  switch (pd) {
    case MXOPT_F32: return plain_pending_for_pd<MXOPT_F32>(gd, g2d, L, lr_p, wd, has_wd, prep);
    case MXOPT_BF16: return plain_pending_for_pd<MXOPT_BF16>(gd, g2d, L, lr_p, wd, has_wd, prep);
    case MXOPT_F16: return plain_pending_for_pd<MXOPT_F16>(gd, g2d, L, lr_p, wd, has_wd, prep);
  }
  return false;
}

bool launch_sgd_plain(int pd, int gd, int od, const Launch& L, float lr_p, float wd, int has_wd, bool g_promoted,
                      const DevPrep& prep) {
  switch (pd) {
    case MXOPT_F32: return plain_for_pd<MXOPT_F32>(gd, od, L, lr_p, wd, has_wd, g_promoted, prep);
    case MXOPT_BF16: return plain_for_pd<MXOPT_BF16>(gd, od, L, lr_p, wd, has_wd, g_promoted, prep);
    case MXOPT_F16: return plain_for_pd<MXOPT_F16>(gd, od, L, lr_p, wd, has_wd, g_promoted, prep);
  }
  return false;
}

// Microseconds without a limit and with it.  Into a buffer of its own: 16-bit into float32 32 M elements 39 and 37, 64 M 74 and
// 68, 256 M 277 and 247, 1.72 G 1,852 and 1,596 (10,000 tensors whose chunks are 82 % full 107 and 122); 16-bit into 16-bit 64 M 49
// and 47, 256 M 182 and 168, 596 M 419 and 374; float32 64 M 93 and 89, 256 M 360 and 351.  Added into a float32 buffer 256 M 435
// and 426, 596 M 1,005 and 954; into a 16-bit one 128 M 131 and 128, 596 M 589 and 553.
// Where the lists' last chunks begin to spoil it (log-uniform lists; per mille full): 16-bit into 16-bit 933 184 and 194, 974 209 and
// 223, 996 317 and 323, the 0.6B list (999) 414 and 371; into float32 933 131 and 137, 961 166 and 168, 984 205 and 203, 996 260 and
// 250; float32 877 141 and 142, 933 178 and 169; added, 16-bit 933 250 and 263, 952 307 and 312, 974 303 and 298, into float32 933 455
// and 438.  In memory of several regions: 16-bit into float32 974 156 and 164, 984 190 and 198, 996 242 and 241, 998 208 and 205; float32
// 933 160 and 165, 952 223 and 223, 974 209 and 206; 16-bit added into float32 256 M 419 and 424, 596 M 935 and 947.
template <int GD, int OD, bool ADD>
constexpr Crowd kTransformCrowd =
    ADD ? (OD == MXOPT_F32 ? (GD == MXOPT_F32 ? kNoLimit : Crowd{2, 900, 256, kNever, 0}) : Crowd{4, 970, 128})
        : (OD != MXOPT_F32 ? Crowd{6, 998, 16} : GD != MXOPT_F32 ? Crowd{4, 970, 16, 995, 16} : Crowd{3, 900, 32, 950, 32});

template <int GD, int OD>
static void launch_transform_t(const Launch& L, const DevPrep& prep, int add) {
  if (L.nontemporal) {
    if (add) MXOPT_LAUNCH_CROWD((transform_kernel<GD, OD, true, true>), (kTransformCrowd<GD, OD, true>), L, prep);
    else MXOPT_LAUNCH_CROWD((transform_kernel<GD, OD, true, false>), (kTransformCrowd<GD, OD, false>), L, prep);
  } else {
    if (add) MXOPT_LAUNCH((transform_kernel<GD, OD, false, true>), L, prep);
    else MXOPT_LAUNCH((transform_kernel<GD, OD, false, false>), L, prep);
  }
}

template <int GD>
static bool transform_for_gd(int od, const Launch& L, const DevPrep& prep, int add) {
  if (od == MXOPT_F32) { launch_transform_t<GD, MXOPT_F32>(L, prep, add); return true; }
  if (od == GD) { launch_transform_t<GD, GD>(L, prep, add); return true; }
  return false;
}

bool launch_transform(int gd, int od, const Launch& L, const DevPrep& prep, int add) {
  switch (gd) {
    case MXOPT_F32: return transform_for_gd<MXOPT_F32>(od, L, prep, add);
    case MXOPT_BF16: return transform_for_gd<MXOPT_BF16>(od, L, prep, add);
    case MXOPT_F16: return transform_for_gd<MXOPT_F16>(od, L, prep, add);
  }
  return false;
}

}  // namespace mxopt
