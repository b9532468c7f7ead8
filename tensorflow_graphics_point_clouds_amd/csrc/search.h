// Cell rows of the sorted grid and the distance test, as the neighbour search and the Poisson-disk
// selection use them.  For files compiled with -ffp-contract=off (the test decides integer output).
#pragma once
#include "common.h"

namespace mccnn {

// Offsets act on dims 0..max(D-2,1); the last dim is covered by the key search.
template <int D>
struct OffsetInfo {
  static constexpr int kDims = (D - 2 > 1 ? D - 2 : 1) + 1;
  static constexpr int count() {
    int c = 1;
    for (int i = 0; i < kDims; ++i) c *= 3;
    return c;
  }
};

inline int offsets_for(int d) {
  int od = (d - 2 > 1 ? d - 2 : 1) + 1, c = 1;
  for (int i = 0; i < od; ++i) c *= 3;
  return c;
}

// Where a cell row's slice of the sorted points is looked for: in `span` of the keys, from the
// first key <= maxk up to the first key < mink.  Nothing left to look for where mink > maxk: the
// slice is `span` itself.
struct KeyRange {
  int2 span;
  int64_t maxk, mink;
};

// The slices of kN cell rows.  The two ends of all of them are searched side by side: a binary
// search is a chain of dependent loads (eleven over 2048 keys), and what one lane has to find is
// kept to one such chain.  Bound by instruction issue as much: an end moves up by steps of falling
// powers of two, which both ends of a row share, for 16 vector instructions a round where bounds
// of each end's own took 30 (763 k centres x 37 pairs 82 -> 79 us; the searches inside the visits
// of a three-level network of 16 x 1024 points 122 -> 108).
template <int kN>
__host__ __device__ __forceinline__ void find_slices(const KeyRange *range,
                                                     const int64_t *__restrict__ keys, int2 *slice) {
  int at[2 * kN], step[kN];
  int open = 0;
#pragma unroll
  for (int i = 0; i < kN; ++i) {
    const int length = range[i].span.y - range[i].span.x;
    const bool search = range[i].mink <= range[i].maxk;
    step[i] = search && length > 0 ? 1 << (31 - __builtin_clz(length)) : 0;
    at[2 * i] = range[i].span.x;
    at[2 * i + 1] = search ? range[i].span.x : range[i].span.y;
    open |= step[i];
  }
  while (open) {
    open = 0;
    int64_t key[2 * kN];
    bool live[2 * kN];
#pragma unroll
    for (int k = 0; k < 2 * kN; ++k) {       // (a step past the end reads a key it ignores)
      // (not the sum against the end: it may pass 2^31 - 1)
      live[k] = step[k / 2] <= range[k / 2].span.y - at[k] && step[k / 2] > 0;
      key[k] = keys[live[k] ? at[k] + step[k / 2] - 1 : 0];
    }
#pragma unroll
    for (int k = 0; k < 2 * kN; ++k) {
      // up to the first key <= maxk, up to the first key < mink
      const bool up = k % 2 == 0 ? key[k] > range[k / 2].maxk : key[k] >= range[k / 2].mink;
      at[k] += live[k] && up ? step[k / 2] : 0;
    }
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      step[i] >>= 1;
      open |= step[i];
    }
  }
#pragma unroll
  for (int i = 0; i < kN; ++i)
    slice[i] = at[2 * i + 1] > at[2 * i] ? make_int2(at[2 * i], at[2 * i + 1]) : make_int2(0, 0);
}

// Whether a candidate lies inside the radius; `live` false: no candidate at all.
template <int D>
__device__ __forceinline__ bool within_radius(bool live, const float *diff, const float *ir) {
  float acc = 0.0f;
#pragma unroll
  for (int d = 0; d < D; ++d) {
    const float sc = diff[d] * ir[d];
    const float sq = sc * sc;
    acc = acc + sq;
  }
  // The reference tests sqrtf(acc) < 1 (count_neighbors_kernels.cu.cc:83-86).  The
  // correctly rounded root is monotonic, sqrtf(1) = 1 and the root of the largest
  // float below 1 is again that float, so acc < 1 decides the same for every
  // float, infinities and NaN included, without the twenty instructions of an
  // IEEE square root per candidate.  (A sum of squares is never below 0.)
  return acc < (live ? 1.0f : 0.0f);
}

}  // namespace mccnn
