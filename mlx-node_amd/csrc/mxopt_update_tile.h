// The optimizer update over long lists, one tile of kTileChunks consecutive chunks at a time.
#pragma once
#include <type_traits>

#include "mxopt_tiles.h"
#include "mxopt_update_chunk.h"

namespace mxopt {

// See mxopt_tiles.h for what a tile gains.  Microseconds by chunks as they were before (parameters' stores plain, as many
// workgroups as fit) and by tiles, plain memory of one region: AdamW of 596 M float32 elements 3,140 and 2,833, bf16 with float32
// moments 2,453 and 2,224, of 1.72 G 7,010 and 6,315, with a float32 buffer and a bf16 micro-batch folded in 8,460 and 7,750; SGD
// with momentum of 1.72 G float32 6,460 and 5,650; RMSprop of 596 M 2,183 and 1,958; plain SGD of 596 M bf16 651 and 585.  What did not help: the parameters stored row by row as they are computed
// (2 % slower: reads and writes mix again), a barrier between the streams' stores, workgroups that stay and walk the tiles
// (4 % slower), tiles that begin at a multiple of their size in memory (nothing on a whole parameter list).
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

// Where tiles begin to pay, in whole tiles per compute unit.  Microseconds by chunks (streaming stores, two workgroups per compute
// unit) and by tiles, memory of one region: float32 AdamW of 128 M elements (16 tiles) 622 and 631, 192 M (24) 948 and 936, 596 M 3,017 and
// 2,874; SGD 128 M 438 and 443, 192 M 659 and 654, 596 M 2,146 and 1,988; bf16 AdamW 256 M (32) 951 and 997, 1.72 G 6,515 and
// 6,301; plain bf16 SGD 256 M 264 and 271, 596 M (71) 592 and 578; a float32 buffer and a bf16 micro-batch folded into AdamW, 596 M
// 2,754 and 2,688.  In memory of two regions the chunks stay ahead by 2 %.
template <int PD, int GD, int G2, class Math>
constexpr uint32_t kUpdateTilesPerCu = (PD == MXOPT_F32 && GD == MXOPT_F32 && G2 <= MXOPT_F32) ? 24 : Math::kV ? 48 : 64;

template <int PD, int GD, int G2, class Math>
static bool launch_update_tiles(const Launch& L, const Math& math, const DevPrep& prep) {
  if (L.ntiles == 0 || !L.in_place || L.tiles_per_cu < kUpdateTilesPerCu<PD, GD, G2, Math>) return false;
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
