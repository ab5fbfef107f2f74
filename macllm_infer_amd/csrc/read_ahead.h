// Weights that the launches behind a launch read, brought into the caches by workgroups of it that do nothing else: a
// launch that waits for round trips leaves the memory idle, and products of few rows are as long as the way of their weights.
#pragma once
#include "common.h"

#define AHEAD_MOST 4

struct AheadWeight {           // as callers give it: tiles one behind the other
  const void* at;
  long tiles, tile_bytes;
};

struct AheadTiles {            // pieces of a tile that a workgroup reads at once, and how far on its next one is
  const void* at;
  int tiles, tile_bytes, pieces, step_tiles, step_pieces;
};

struct AheadList {
  AheadTiles weight[AHEAD_MOST];
};

// `blocks` (a multiple of 8) workgroups of `threads` threads; false: a weight that is none, or too large for the numbers.
static inline bool read_ahead_list(AheadList& list, const AheadWeight* weights, int count, int blocks, int threads) {
  if (count < 0 || count > AHEAD_MOST || (count && !weights)) return false;
  for (int k = 0; k < AHEAD_MOST; ++k) {
    list.weight[k] = {nullptr, 0, 16, 1, 0, 0};
    if (k >= count) continue;
    const AheadWeight& w = weights[k];
    if (!w.at || (uintptr_t)w.at % 16 || w.tiles <= 0 || w.tile_bytes <= 0 || w.tile_bytes % 16 || w.tiles > (1 << 28) || w.tile_bytes > (1 << 28))
      return false;
    const int pieces = (int)((w.tile_bytes + threads * 16 - 1) / (threads * 16)), peers = blocks / 8;
    list.weight[k] = {w.at, (int)w.tiles, (int)w.tile_bytes, pieces, peers / pieces, peers % pieces};
  }
  return true;
}

// Workgroup `block` of those that read ahead.  What it leaves is in the caches: a tile is read on the die whose cache the
// product's workgroup of that number will ask (workgroups go to the eight dies in turn), or, where other bytes have pushed it
// out, in the memory-side cache.  Pieces of THREADS 16-byte words, dealt out to the die's workgroups in the order in which
// the products will read them.
template <int THREADS>
__device__ __forceinline__ void read_ahead_block(const AheadList& list, int block) {
  const int die = blockIdx.x % 8, first = block / 8;
  constexpr int PIECE = THREADS * 16;
#pragma unroll
  for (int k = 0; k < AHEAD_MOST; ++k) {
    const AheadTiles w = list.weight[k];
    const int tiles = (w.tiles - die + 7) / 8;                           // of this die
    int tile = first / w.pieces, piece = first - tile * w.pieces;
    while (tile < tiles) {
      uint4 word[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int at = min(piece * PIECE + (int)threadIdx.x * 16, w.tile_bytes - 16);
        word[j] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(w.at) + (long)(die + 8 * min(tile, tiles - 1)) * w.tile_bytes + at);
        tile += w.step_tiles;
        piece += w.step_pieces;
        if (piece >= w.pieces) {
          piece -= w.pieces;
          ++tile;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) asm volatile("" ::"v"(word[j].x), "v"(word[j].y), "v"(word[j].z), "v"(word[j].w));
    }
  }
}
