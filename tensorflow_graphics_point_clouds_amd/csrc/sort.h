// The radix sort of sort.hip as the grid uses it.
#pragma once
#include "common.h"

namespace mccnn {

constexpr int kSortThreads = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr int kSortWaves = kSortThreads / kWave;
constexpr int kSortRadix = 256;

struct SortWorkspace {
  int64_t *keys_tmp;   // [n]
  int *idx_tmp;        // [n]
  int *hist;           // [256][tiles]
  int *totals;         // [256]
  size_t bytes;
};

SortWorkspace carve_sort_workspace(void *ws, int64_t n);

// What the last pass gathers along with the order.
struct SortedPoints {
  const float *points;
  const int *batch_ids;
  float *points_out;
  int *batch_ids_out;
};

// Stable descending sort of 32-bit keys of `bits` significant bits; w.hist already holds the
// digit histogram of the first pass ([digit][tile of kSortTile keys]).  keys32 is overwritten.
int sort_grid_keys(hipStream_t s, int num_dims, int64_t n, int bits, unsigned *keys32,
                   const SortWorkspace &w, int64_t *keys_out, int *idx_out, const SortedPoints &g);

// Order of 32-bit keys, descending and stable; keys32 is overwritten.
int sort_order32(hipStream_t s, int64_t n, unsigned *keys32, const SortWorkspace &w, int *idx_out);

}  // namespace mccnn
