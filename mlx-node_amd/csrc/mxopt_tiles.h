// Building blocks of the tiled kernels: one workgroup of 1,024 lanes per tile of kTileChunks consecutive chunks.
//
// What bounds the passes that read and write is how often the memory has to turn round between the two, and how much of a
// row it moves in between.  A chunk's workgroup writes 8 or 16 KB of one stream, then of the next, while its three or more
// neighbours on the compute unit are in other phases.  A tile's workgroup is alone on its compute unit, loads its streams one
// after the other and stores them one after the other: runs of 64 KB of a 16-bit stream and 128 KB of a float32 one where a lane's
// registers hold the whole tile, half of that in two turns where they do not.  In memory of one region (where a plain allocation
// lies) a long list of several streams reaches 5.8 - 6.1 TB/s by tiles, 5.6 - 6.1 by chunks with few workgroups per compute unit, 5.3 -
// 5.6 with many; in memory of two regions 6.2 - 6.35 by tiles, 6.3 - 6.45 by chunks.
// Bare streams, 4 read and 3 written, float32, 596 M elements: 256 lanes x 16 elements 3,150 us, 1,024 x 16 in the same
// order 3,160, stream by stream 2,850; 512 x 32 3,050; 1,024 x 8 3,190.  Two 16-bit streams and two float32 ones: 2,490 by chunks,
// 1,024 x 16 2,350, 1,024 x 32 2,140.
#pragma once
#include "mxopt_kernels_common.h"

namespace mxopt {

constexpr int kTileThreads = 1024;

// Four elements as they lie in memory.
template <int DT>
struct Piece {
  using T = u32x2;
  using Mem = u32x2_mem;
  static __device__ __forceinline__ void unpack(const T& r, float (&x)[4]) {
    x[0] = Elem<DT>::unpack(r.x & 0xffffu); x[1] = Elem<DT>::unpack(r.x >> 16);
    x[2] = Elem<DT>::unpack(r.y & 0xffffu); x[3] = Elem<DT>::unpack(r.y >> 16);
  }
  static __device__ __forceinline__ T pack(const float (&x)[4]) {
    return T{Elem<DT>::pack2(x[0], x[1]), Elem<DT>::pack2(x[2], x[3])};
  }
};
template <>
struct Piece<MXOPT_F32> {
  using T = f32x4;
  using Mem = f32x4_mem;
  static __device__ __forceinline__ void unpack(const T& r, float (&x)[4]) { x[0] = r.x; x[1] = r.y; x[2] = r.z; x[3] = r.w; }
  static __device__ __forceinline__ T pack(const float (&x)[4]) { return T{x[0], x[1], x[2], x[3]}; }
};

// Lane `tid`'s piece of row `first` of a stream.  The row's address is the same for the whole workgroup; pinned to scalar
// registers the access takes it as its scalar base and needs one 32-bit lane offset for all rows (the compiler would
// otherwise keep a 64-bit vector address for each of the tile's rows and streams).
template <int DT>
__device__ __forceinline__ MXOPT_GLOBAL typename Piece<DT>::Mem* piece_address(const void* stream, uint64_t first, uint32_t tid) {
  uintptr_t row = (uintptr_t)stream + first * Elem<DT>::kBytes;
  uint32_t lane = tid * (4u * Elem<DT>::kBytes);
  asm("" : "+s"(row));
  asm("" : "+v"(lane));
  return (MXOPT_GLOBAL typename Piece<DT>::Mem*)((MXOPT_GLOBAL char*)row + lane);
}
template <int DT, bool NT>
__device__ __forceinline__ typename Piece<DT>::T load_piece(const void* stream, uint64_t first, uint32_t tid) {
  const MXOPT_GLOBAL typename Piece<DT>::Mem* q = piece_address<DT>(stream, first, tid);
  const typename Piece<DT>::T r = NT ? __builtin_nontemporal_load(q) : *q;
  __builtin_amdgcn_sched_barrier(0);  // in program order: the rows are waited for in the order they are computed in
  return r;
}
template <int DT, bool NT>
__device__ __forceinline__ void store_piece(void* stream, uint64_t first, uint32_t tid, const typename Piece<DT>::T& r) {
  MXOPT_GLOBAL typename Piece<DT>::Mem* q = piece_address<DT>(stream, first, tid);
  const typename Piece<DT>::Mem m = r;
  if (NT) __builtin_nontemporal_store(m, q); else *q = m;
}

template <class T>
__device__ __forceinline__ void pin(T& piece) {
  asm volatile("" : "+v"(piece));
}

// The workgroup's tile and the descriptor of its first chunk's tensor.
struct TileView {
  DevTile tile;
  DevTensor t;
  bool whole;
};
__device__ __forceinline__ TileView this_tile(const DevTensor* __restrict__ T, const DevTensor& one, uint32_t nchunks,
                                              const DevTile* __restrict__ tiles) {
  TileView tv;
  if (tiles != nullptr) {
    tv.tile = load_constant<DevTile>(tiles, blockIdx.x);
    tv.t = load_constant<DevTensor>(T, tv.tile.tensor);
    tv.whole = (tv.tile.count & kTileWhole) != 0;
    tv.tile.count &= ~kTileWhole;
  } else {  // a single tensor described in the kernel arguments
    tv.t = one;
    const uint32_t entry = blockIdx.x * kTileChunks;
    tv.tile = DevTile{entry, nchunks - entry < kTileChunks ? nchunks - entry : kTileChunks, 0u, entry};
    tv.whole = entry + kTileChunks <= (uint32_t)((one.n - one.head) >> 12);
  }
  return tv;
}

// Calls chunk(view, lane) for each chunk of a tile that is not whole, four at a time.
template <class F>
__device__ __forceinline__ void chunks_of_tile(const DevTensor* __restrict__ T, const DevChunk* __restrict__ C, const DevTensor& one,
                                               const DevTile& tile, F&& chunk) {
  for (uint32_t k = __builtin_amdgcn_readfirstlane(threadIdx.x / kThreads); k < tile.count; k += kTileThreads / kThreads)
    chunk(locate(T, C, one, tile.entry + k), threadIdx.x % kThreads);
}

#define MXOPT_ROWS _Pragma("unroll") for (int j = 0; j < U; ++j)

// Dynamic LDS of every tiled launch, unused: more than half a compute unit's 160 KB, so that one workgroup has it to itself.
// Plain SGD on 596 M bf16 elements: 586 us with it, 659 without (AdamW's registers have the same effect).  Kernels of another stream
// find less room meanwhile: ten float32 AdamW updates of 256 M and matrix products of 8,192 on another stream, 12.4 and 8.0 ms alone,
// take 20.4 ms together, 19.4 with the chunk kernel as it was without limits (13.4 alone); with products of 4,096 18.7 and 21.3.
constexpr unsigned kOnePerCu = 84 * 1024;

}  // namespace mxopt
