// Stable descending sort of up to 16 384 keys by one block of 16 wavefronts, in registers and
// LDS: the sort of a small cloud, for kernels that have the keys at hand.
//
// A launch on this device costs as much as sorting a few thousand keys, so the whole sort is one
// block: LSD passes over digits of up to 10 bits (the digits share the key's bits evenly: 17
// bits are two passes of 9, where 8-bit digits take three).  Wavefront w owns the w-th
// sixteenth of the items, 16 per lane, as their indices; a pass fetches the digits of its items
// from the keys in memory (L2; keys carried along in registers and exchanged through LDS spill).
// Per pass: digit counts per wavefront with LDS atomics (counts do not depend on the order), a
// block scan over (digit, wavefront), then every wavefront ranks its items in rounds of 64 in
// input order -- the rank among the lanes with the same digit comes from ballots, the first such
// lane advances the wavefront's position -- and the indices change places through LDS.  No
// atomics in the ranking: the order is stable and deterministic.
// Bound by instruction issue of one compute unit (about 60 vector instructions per round and
// pass in the ranking), not by memory.
#pragma once
#include "common.h"

namespace mccnn {

constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / kWave;
constexpr int kSmallRounds = 16;                          // keys per lane
constexpr int kSmallMax = kSmallThreads * kSmallRounds;
constexpr int kSmallDigitBits = 10;

struct SmallSortLds {
  int start[kSmallWaves << kSmallDigitBits];              // [wavefront][digit] counts, then positions
  unsigned short exchange[kSmallMax];
  int wave_total[kSmallWaves];
};

// Position of a lane's r-th item: first + 64 r + lane.
__device__ __forceinline__ int small_first(int n) {
  const int per_wave = ((n + kSmallWaves - 1) / kSmallWaves + kWave - 1) / kWave * kWave;
  const int first = (threadIdx.x / kWave) * per_wave;
  return first < n ? first : n;
}
__device__ __forceinline__ int small_last(int n) {
  const int per_wave = ((n + kSmallWaves - 1) / kSmallWaves + kWave - 1) / kWave * kWave;
  const int last = (threadIdx.x / kWave + 1) * per_wave;
  return last < n ? last : n;
}

// item[r] of a lane becomes the index of the key with rank first + 64 r + lane.  `keys` must be
// visible to the whole block (a barrier since they were written); the lowest `bits` of keys less
// `below` tell them apart.  kRounds: n <= 1024 kRounds (the loops over rounds are unrolled and
// cost their instructions whether a round has items or not).
template <int kRounds>
__device__ __forceinline__ void small_sort(int n, int bits, const int64_t *keys, int64_t below,
                                           int *item, SmallSortLds &s) {
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int first = small_first(n), last = small_last(n);
  const int passes = (bits + kSmallDigitBits - 1) / kSmallDigitBits;
  const int width = (bits + passes - 1) / passes;
  const int radix = 1 << width;
#pragma unroll
  for (int r = 0; r < kRounds; ++r) item[r] = first + r * kWave + lane;
  for (int p = 0; p < passes; ++p) {
    const int shift = p * width;
    int digit[kRounds];
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
      digit[r] = first + r * kWave + lane < last
                     ? (int)((~(uint64_t)(keys[item[r]] - below) >> shift) & (uint64_t)(radix - 1)) : 0;
    for (int i = t; i < kSmallWaves * radix; i += kSmallThreads) s.start[i] = 0;
    __syncthreads();
    int *mine = s.start + wave * radix;
#pragma unroll
    for (int r = 0; r < kRounds; ++r)
      if (first + r * kWave + lane < last) atomicAdd(&mine[digit[r]], 1);
    __syncthreads();
    // thread t scans digit t over the wavefronts, the block scans the digits
    int total = 0;
    if (t < radix)
#pragma unroll
      for (int w = 0; w < kSmallWaves; ++w) total += s.start[w * radix + t];
    const int incl = wave_inclusive_scan(total);
    if (lane == kWave - 1) s.wave_total[wave] = incl;
    __syncthreads();
    int run = incl - total;
    for (int w = 0; w < wave; ++w) run += s.wave_total[w];
    if (t < radix)
      for (int w = 0; w < kSmallWaves; ++w) {
        const int c = s.start[w * radix + t];
        s.start[w * radix + t] = run;
        run += c;
      }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      __builtin_amdgcn_sched_barrier(0);                  // rounds one after another: few registers
      if (first + r * kWave < last) {                     // uniform in the wavefront
        const bool live = first + r * kWave + lane < last;
        const int d = digit[r];
        uint64_t same = __ballot(live);
        for (int bit = 0; bit < width; ++bit) {
          const uint64_t b = __ballot((d >> bit) & 1);
          same &= ((d >> bit) & 1) ? b : ~b;
        }
        const int below = __popcll(same & ((1ull << lane) - 1ull));
        int dst = 0;
        if (live) dst = mine[d] + below;
        wave_lds_sync();                                  // every lane has read its position
        if (live && below == 0) mine[d] = dst + __popcll(same);
        if (live) s.exchange[dst] = (unsigned short)item[r];
        wave_lds_sync();
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kRounds; ++r) {
      const int i = first + r * kWave + lane;
      if (i < last) item[r] = s.exchange[i];
    }
  }
}

__device__ __forceinline__ void small_sort_any(int n, int bits, const int64_t *keys, int64_t below,
                                               int *item, SmallSortLds &s) {
  if (n <= kSmallThreads) small_sort<1>(n, bits, keys, below, item, s);
  else if (n <= 4 * kSmallThreads) small_sort<4>(n, bits, keys, below, item, s);
  else small_sort<kSmallRounds>(n, bits, keys, below, item, s);
}

}  // namespace mccnn
