// Tiles of a step's tokens, found on the device: the tokens of every request that brings `from` or more are cut into tiles
// of up to `size`, tiles counted through these requests in order.  Called by whole waves.
#pragma once
#include "common.h"

struct TokenTile {
  int req, tile;      // the request (-1: there is no such tile) and the tile's number within it; the same in every lane
};

__device__ inline int token_tiles(int tokens, int size, int from) { return tokens >= from ? (tokens + size - 1) / size : 0; }

__device__ inline TokenTile find_token_tile(const int* __restrict__ q_start, int R, int size, int wanted, int from = 1) {
  const int lane = threadIdx.x % PI_WAVE;
  int tile = wanted, req = -1;
  for (int r0 = 0; r0 < R; r0 += PI_WAVE) {
    const int r = r0 + lane;
    const int mine = r < R ? token_tiles(q_start[r + 1] - q_start[r], size, from) : 0;
    int upto = mine;
#pragma unroll
    for (int d = 1; d < PI_WAVE; d *= 2) {
      const int other = __shfl_up(upto, d, PI_WAVE);
      if (lane >= d) upto += other;
    }
    const unsigned long long past = __ballot(upto > tile);
    if (past) {
      const int at = __ffsll(past) - 1;
      req = r0 + at;
      tile -= __shfl(upto - mine, at, PI_WAVE);
      break;
    }
    tile -= __shfl(upto, PI_WAVE - 1, PI_WAVE);
  }
  return TokenTile{__builtin_amdgcn_readfirstlane(req), __builtin_amdgcn_readfirstlane(tile)};
}

// Tiles of the requests before `req`.
__device__ inline int token_tiles_before(const int* __restrict__ q_start, int req, int size, int from = 1) {
  int sum = 0;
  for (int r = threadIdx.x % PI_WAVE; r < req; r += PI_WAVE) sum += token_tiles(q_start[r + 1] - q_start[r], size, from);
#pragma unroll
  for (int d = PI_WAVE / 2; d > 0; d /= 2) sum += __shfl_xor(sum, d, PI_WAVE);
  return __builtin_amdgcn_readfirstlane(sum);
}
