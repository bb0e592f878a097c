// radix_tile.hpp -- the stable order of a workgroup's tile by a digit of its
// keys, shared by the radix sort and by the column sums' last digit.
#pragma once

#include "common.hpp"

namespace tbsla_hip {

constexpr int kRadix = 256;

// Places of a tile's elements in digit order.  A thread holds elements
// sub + i * kWave (sub below), those before count counting; pos[i] is element i's
// place in the tile, and start and total, in thread d, are digit d's first place
// and its elements.
template <int THREADS>
struct TileRank {
  int wcnt[THREADS / kWave][kRadix];  // counts, then each wave's first position
  int gofs[kRadix];                   // for the caller
  int wsum[THREADS / kWave];
};

// this lane's first element of the tile
template <int ITEMS>
__device__ inline int tile_sub() {
  return threadIdx.x / kWave * kWave * ITEMS + (threadIdx.x & (kWave - 1));
}

template <int THREADS, int ITEMS, typename K>
__device__ inline void rank_tile(TileRank<THREADS> &sh, const K (&key)[ITEMS], int (&pos)[ITEMS],
                                 int count, int shift, int bits, int &start, int &total) {
  constexpr int waves = THREADS / kWave;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int mask = (1 << bits) - 1, sub = tile_sub<ITEMS>();
  for (int i = threadIdx.x; i < waves * kRadix; i += THREADS) (&sh.wcnt[0][0])[i] = 0;
  __syncthreads();
  // rank of every element among its wave's elements of the same digit
  const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
#pragma unroll
  for (int i = 0; i < ITEMS; i++) {
    if (sub - lane + i * kWave >= count) break;  // the whole wave's
    const bool valid = sub + i * kWave < count;
    const int d = (int)(key[i] >> shift) & mask;
    unsigned long long peers = __ballot(valid);
    for (int b = 0; b < bits; b++) {
      const bool bit = (d >> b) & 1;
      const unsigned long long m = __ballot(bit);
      peers &= bit ? m : ~m;
    }
    const int rank = __popcll(peers & below);
    const int before = valid ? sh.wcnt[wave][d] : 0;
    pos[i] = before + rank;
    __builtin_amdgcn_wave_barrier();
    if (valid && rank == 0) sh.wcnt[wave][d] = before + __popcll(peers);
    __builtin_amdgcn_wave_barrier();
  }
  __syncthreads();
  // digit starts within the tile (exclusive scan over digits), wave starts
  // within each digit; thread d < kRadix owns digit d
  int incl = 0;
  total = 0;
  if (threadIdx.x < kRadix) {
    for (int w = 0; w < waves; w++) {
      const int c = sh.wcnt[w][threadIdx.x];
      sh.wcnt[w][threadIdx.x] = total;
      total += c;
    }
    incl = total;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
      const int o = __shfl_up(incl, off, kWave);
      if (lane >= off) incl += o;
    }
    if (lane == kWave - 1) sh.wsum[wave] = incl;
  }
  __syncthreads();
  if (threadIdx.x < kRadix) {
    start = incl - total;
    for (int w = 0; w < wave; w++) start += sh.wsum[w];
    for (int w = 0; w < waves; w++) sh.wcnt[w][threadIdx.x] += start;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITEMS; i++)
    if (sub + i * kWave < count) pos[i] += sh.wcnt[wave][(int)(key[i] >> shift) & mask];
}

}  // namespace tbsla_hip
