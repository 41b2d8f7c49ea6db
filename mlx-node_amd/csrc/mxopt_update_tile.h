// The optimizer update over long lists, one tile of kTileChunks consecutive chunks at a time.
#pragma once
#include <type_traits>

#include "mxopt_tiles.h"
#include "mxopt_update_chunk.h"

namespace mxopt {

// See mxopt_tiles.h for what a tile gains, and update_tiles_per_cu for where.  What did not help: the parameters stored row by row
// as they are computed (2 % slower: reads and writes mix again), a barrier between the streams' stores, workgroups that stay and
// walk the tiles (4 % slower), tiles that begin at a multiple of their size in memory (nothing on a whole parameter list).
//
// U rows of 4,096 elements are in registers at once: 8 (the tile) while a row takes at most 12 of them a lane, else 4 in two
// turns (8 would not fit the 128 that 1,024 lanes leave each).
template <int PD, int GD, int G2, class Math, int U>
__global__ __launch_bounds__(kTileThreads) void update_tile_kernel(const DevTensor* __restrict__ T,
                                                                   const DevChunk* __restrict__ C, DevTensor one,
                                                                   uint32_t nchunks, const DevTile* __restrict__ tiles,
                                                                   Math math, DevPrep prep) {
  constexpr bool NT = true;
  using Gradient = GradientOf<GD, G2>;
  constexpr bool kHasG2 = Gradient::kHasG2;
  constexpr int G2D = Gradient::G2D;
  if (skip_requested(prep)) return;
  const PrepRegs pr = load_prep(prep);
  const uint32_t tid = threadIdx.x;

  const TileView tv = this_tile(T, one, nchunks, tiles);
  if (!tv.whole) {
    chunks_of_tile(T, C, one, tv.tile, [&](const ChunkView& cv, uint32_t lane) {
      update_chunk<PD, GD, PD, G2, Math, NT, NT>(cv, lane, math, pr);
    });
    return;
  }
  const DevTensor& t = tv.t;
  const uint32_t flags = t.flags;
  const float bc1 = t.bc1, bc2 = t.bc2;
  const bool use_v = math.uses_v(flags), read_v = math.reads_v(flags);
#pragma unroll 1
  for (uint32_t h = 0; h < kTileChunks / U; ++h) {
    const uint64_t first = t.head + (uint64_t)(tv.tile.index + h * U) * kChunk;
    typename Piece<PD>::T p[U];
    typename Piece<GD>::T g[U];
    typename Piece<G2D>::T g2[U];
    f32x4 m[U], v[U];
    MXOPT_ROWS g[j] = load_piece<GD, NT>(t.g, first + j * kChunk, tid);
    if (kHasG2) { MXOPT_ROWS g2[j] = load_piece<G2D, NT>(t.g_out, first + j * kChunk, tid); }
    MXOPT_ROWS p[j] = load_piece<PD, NT>(t.p, first + j * kChunk, tid);
    if (Math::kM) { MXOPT_ROWS m[j] = load_piece<MXOPT_F32, NT>(t.m, first + j * kChunk, tid); }
    if (Math::kV) {
      if (read_v) { MXOPT_ROWS v[j] = load_piece<MXOPT_F32, NT>(t.v, first + j * kChunk, tid); }
      else { MXOPT_ROWS v[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }
    }
    // Row by row: computed side by side the rows would not fit the registers.  The empty statements in front of a row's
    // arithmetic and behind it are what keeps the compiler from moving any of it to another row.
    MXOPT_ROWS {
      pin(p[j]); pin(g[j]);
      if (kHasG2) pin(g2[j]);
      if (Math::kM) pin(m[j]);
      if (Math::kV) pin(v[j]);
      float xp[4], xg[4], xg2[4], xm[4], xv[4];
      Piece<PD>::unpack(p[j], xp);
      Piece<GD>::unpack(g[j], xg);
      if (kHasG2) Piece<G2D>::unpack(g2[j], xg2);
      if (Math::kM) Piece<MXOPT_F32>::unpack(m[j], xm);
      if (Math::kV) Piece<MXOPT_F32>::unpack(v[j], xv);
      if (pr.flags != 0) Gradient::template combine_row<true>(pr, xg, xg2);
      else Gradient::template combine_row<false>(pr, xg, xg2);
      float sq[4] = {};
      if constexpr (Math::kSquare) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float s = math.squared(xp[e], xg[e]);
          sq[e] = s * s;
        }
        if (GD != MXOPT_F32 && math.rounds_square()) round_group<GD, 4>(sq);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) math.apply(xp[e], xg[e], xm[e], xv[e], bc1, bc2, flags, sq[e]);
      p[j] = Piece<PD>::pack(xp);
      if (Math::kM) m[j] = Piece<MXOPT_F32>::pack(xm);
      if (Math::kV) v[j] = Piece<MXOPT_F32>::pack(xv);
      pin(p[j]);
      if (Math::kM) pin(m[j]);
      if (Math::kV) pin(v[j]);
    }
    __builtin_amdgcn_sched_barrier(0);
    MXOPT_ROWS store_piece<PD, NT>(t.p_out, first + j * kChunk, tid, p[j]);
    __builtin_amdgcn_sched_barrier(0);
    if (Math::kM) { MXOPT_ROWS store_piece<MXOPT_F32, NT>(t.m, first + j * kChunk, tid, m[j]); }
    __builtin_amdgcn_sched_barrier(0);
    if (use_v) { MXOPT_ROWS store_piece<MXOPT_F32, NT>(t.v, first + j * kChunk, tid, v[j]); }
  }
  if (tv.tile.index == 0 && tid < t.head) {  // elements in front of the first aligned group
    ChunkView head = locate(T, C, one, tv.tile.entry);
    head.fast = false;
    head.len = 0;
    update_chunk<PD, GD, PD, G2, Math, NT, NT>(head, tid, math, pr);
  }
}

// Where tiles begin to pay in memory of one region, in whole tiles per compute unit.  Microseconds by chunks and by tiles, pairs
// from several places in memory: float32 AdamW of 192 M elements (24 tiles) 946 and 942, 909 and 914, 596 M 2,850 and 2,828, 2,658 and
// 2,691, 310 M in 4,000 tensors 1,451 and 1,428; SGD 192 M 642 and 647, 660 and 653, 1.5 G 5,544 and 5,239, 5,408 and 5,293, the 4,000 tensors
// 1,077 and 1,052; plain SGD 192 M 398 and 399, the 4,000 648 and 609.  A float32 buffer and a bf16 micro-batch folded into bf16 AdamW 384 M
// (48) 1,813 and 1,749, 1.72 G 7,885 and 7,729, 7,490 and 7,351, into plain SGD 512 M (64) 907 and 883; SGD and RMSprop of 16-bit
// parameters 384 M 967 and 919, 958 and 908, 945 and 917, 950 and 909.  bf16 AdamW 512 M 1,938 and 2,027, 1 G
// (127) 4,046 and 4,029, 3,739 and 3,833, 1.72 G (205) 6,316 and 6,328 (means of five), behind its norm with several lists in turn
// 7,028 and 6,868; plain bf16 SGD 512 M 524 and 533, 596 M (71) 587 and 585, behind its norm 815 and 801.  Never ahead: float32 RMSprop
// 192 M 644 and 668, 1.72 G 5,554 and 5,661.
template <int PD, int GD, int G2, class Math>
constexpr uint32_t update_tiles_per_cu() {
  constexpr uint32_t kNoLength = 0xffffffffu - 1u;  // option "tiles" = 2 says 0xffffffff
  if (PD == MXOPT_F32 && GD == MXOPT_F32 && G2 <= MXOPT_F32) return Math::kSquare && !Math::kM ? kNoLength : 24u;
  if (!Math::kV) return 64u;
  return Math::kM && G2 < 0 ? 192u : 48u;
}

template <int PD, int GD, int G2, class Math>
static bool launch_update_tiles(const Launch& L, const Math& math, const DevPrep& prep) {
  if (L.ntiles == 0 || !L.in_place || L.tiles_per_cu < update_tiles_per_cu<PD, GD, G2, Math>()) return false;
  constexpr int kG2Words = G2 < 0 ? 0 : Elem<(G2 < 0 ? MXOPT_F32 : G2)>::kBytes;
  constexpr int kWords = Elem<PD>::kBytes + Elem<GD>::kBytes + kG2Words + (Math::kM ? 4 : 0) + (Math::kV ? 4 : 0);
  constexpr int U = kWords <= 12 ? 8 : 4;
  hipLaunchKernelGGL((update_tile_kernel<PD, GD, G2, Math, U>), dim3(L.ntiles), dim3(kTileThreads),
                     note_launch(L, kTileThreads, L.ntiles, kOnePerCu), L.stream, L.tensors, L.chunks, L.one, L.nchunks,
                     L.tiles, math, prep);
  if (L.note != nullptr) L.note->streams_parameters = 1;
  return true;
}

}  // namespace mxopt
