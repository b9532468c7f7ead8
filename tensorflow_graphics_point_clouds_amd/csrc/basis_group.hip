// Gradients of the basis projection with the scatter-add of the feature gradient gathered in LDS
// per group of centres that share their points
// (custom_ops/tfg_custom_ops/basis_proj/cc/kernels/basis_proj_grads_kernels.cu.cc:29-151):
//   dbasis[m,k]  = sum_c g[i,c,k] * feat[nbr_m, c]
//   dfeat[n,c]  += sum_k g[i,c,k] * basis[m,k]               (n = nbr_m, i = centre of m)
//
// With one atomic per pair and channel the scatter is bound by the atomic units: 43.7 M pairs x
// 128 channels at 328 G adds/s are 17 of the 22.8 ms the kernel of basis_proj.hip takes.  Centres
// that lie close together list mostly the same points, so a block takes a group of them, adds
// the rows of its pairs up in an LDS table keyed by point, and sends every row out once.  LDS
// float atomics are no way to do that (200 G adds/s over the device, slower than memory's);
// plain reads and writes are (2100 G/s), so every wavefront owns 16 channels of the table and
// walks all pairs of the group for them -- no two wavefronts touch the same word, and the pairs
// of one centre list distinct points (a point listed twice is noticed when the points are
// numbered and takes the atomic).
//
// The caller's order of the centres is arbitrary; which of them are neighbours is found from the
// table itself: centres ordered by the smallest hash of their points (and a second one) bring
// those with overlapping lists together, whatever the numbering (3.9 pairs per point at 16
// centres of 52 pairs, against 4.3 in the order of the grid's cells).
//
// Measured (both gradients, order of the centres included), one atomic per pair and channel ->
// grouped: 800 k points x 52 pairs, 128 channels x 32: 22.8 -> 13.3 ms by one kernel for both (15.1 by
// one for either, dbasis 5.3 and dfeat 9.4); shapes without a matrix-core kernel in
// basis_proj.hip: 200 k x 30, 128 x 64: 66 -> 5.2 ms; 400 k x 30, 96 x 16: 19.1 -> 3.8 ms; 100 k x
// 20, 24 x 8 and 3 x 32: 1.16 -> 0.34, 1.81 -> 0.36 ms.
#include <type_traits>

#include "common.h"
#include "fill.h"
#include "group_walk.h"
#include "mfma.h"
#include "sort.h"

namespace mccnn {

// Pairs of a table, at most: the kernels step through a centre's pairs in 32 bits and look up to two
// chunks (128 pairs) past the last of them.
constexpr int64_t kMostPairs = ((int64_t)1 << 31) - 1024;

// The finalizer "lowbias32" of C. Wellons' hash prospector (public domain).
__device__ __forceinline__ unsigned hash_id(unsigned x) {
  x ^= x >> 16; x *= 0x7feb352du;
  x ^= x >> 15; x *= 0x846ca68bu;
  return x ^ (x >> 16);
}

// ---------------------------------------------------------------- order of centres ----

// 8 lanes per centre: the smallest and the smallest second hash of its points as one key.  The
// smaller half of the bits of a minimum over tens of hashes is not used: 24 bits tell the
// minima apart, 8 of the second order the centres that share one.
__global__ void __launch_bounds__(256) neighbourhood_key_kernel(int64_t n,
                                                                const int2 *__restrict__ nbrs,
                                                                const int *__restrict__ ranges,
                                                                unsigned *__restrict__ keys) {
  const int64_t c = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 3;
  if (c >= n) return;
  const int sub = threadIdx.x & 7;
  const int a = c > 0 ? ranges[c - 1] : 0, b = ranges[c];
  unsigned m1 = 0xffffffffu, m2 = 0xffffffffu;
  for (int m = a + sub; m < b; m += 8) {
    const unsigned h = hash_id((unsigned)nbrs[m].x);
    m1 = h < m1 ? h : m1;
    const unsigned h2 = h * 0x9e3779b1u;
    m2 = h2 < m2 ? h2 : m2;
  }
#pragma unroll
  for (int off = 4; off > 0; off >>= 1) {
    const unsigned o1 = __shfl_xor(m1, off, kWave), o2 = __shfl_xor(m2, off, kWave);
    m1 = o1 < m1 ? o1 : m1;
    m2 = o2 < m2 ? o2 : m2;
  }
  if (sub == 0) keys[c] = (m1 & 0xffffff00u) | ((m2 >> 20) & 0xffu);
}

// --------------------------------------------------------------------- dbasis ----

// dbasis^T [k x pair] = G^T [k x c] F^T [c x pair] on the matrix cores, one wavefront per
// centre: G in registers, the feature rows in tiles of 16 pairs through LDS.  A matrix
// instruction wants pair `col` in lane `col`, a row per lane; loads of that shape touch 64 lines
// and take the address unit 65 cycles for a kilobyte instead of 17 (measured), so the rows are
// fetched in runs of consecutive lanes, one tile ahead, and turned in LDS (rows padded by one
// 16-byte piece: reads of a column of pieces fall into different banks).  The reduction runs
// over channels 16 j + 4 quarter + e (step 4 j + e), a 16-byte read per lane and j.
// Centres go by `order` with neighbours on one XCD, so that most rows come from its L2
// (800 k x 52 pairs, 128 x 32: 5.40 -> 5.29 ms).
template <int CT, int K, bool kFull>
__global__ void __launch_bounds__(256) basis_grads_kernel(
    int64_t n_out, int C, const float *__restrict__ feat, const int2 *__restrict__ nbrs,
    const int *__restrict__ ranges, const int *__restrict__ order,
    const float *__restrict__ in_grad, float *__restrict__ dbasis) {
  constexpr int KT = K > 16 ? K / 16 : 1;
  constexpr int kPieces = 4 * CT, kLd = kPieces + 1;      // 16-byte pieces of a row
  __shared__ v4f tiles[kWavesPerBlock][16 * kLd];
  const int lane = lane_id(), quarter = lane >> 4, col = lane & 15;
  v4f *tile = tiles[threadIdx.x / kWave];
  const int64_t slot = wave_slot_xcd();
  if (slot >= n_out) return;
  const int64_t centre = centre_of(slot, order);
  const int a = centre > 0 ? ranges[centre - 1] : 0, b = ranges[centre];
  if (b <= a) return;
  auto pair_ids = [&](int m0) { return nbrs[m0 + lane < b ? m0 + lane : b - 1].x; };
  int ids = 0, ids_next = pair_ids(a);
  const float *gi = in_grad + centre * (int64_t)C * K;
  float gk[4 * CT][KT];
#pragma unroll
  for (int j = 0; j < CT; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        const int c = 16 * j + 4 * quarter + e;
        gk[4 * j + e][kt] =
            (kFull || c < C) && (K >= 16 || col < K) ? gi[c * K + 16 * kt + col] : 0.0f;
      }
  v4f f[CT];
  auto fetch = [&](int m0) {            // the rows of pairs [m0, m0 + 16)
    if (((m0 - a) & 63) == 0) {
      ids = ids_next;
      ids_next = pair_ids(m0 + 64);
    }
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int i = 64 * j + lane, row = i / kPieces, c = 4 * (i - row * kPieces);
      const float *src = feat + (int64_t)__shfl(ids, ((m0 - a) & 63) + row, kWave) * C + c;
      if constexpr (kFull) {
        f[j] = *reinterpret_cast<const v4f *>(src);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) f[j][e] = c + e < C ? src[e] : 0.0f;
      }
    }
  };
  fetch(a);
  for (int m0 = a; m0 < b; m0 += 16) {
    wave_lds_sync();                    // the tile before has been read
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const int i = 64 * j + lane, row = i / kPieces;
      tile[row * kLd + i - row * kPieces] = f[j];
    }
    wave_lds_sync();
    if (m0 + 16 < b) fetch(m0 + 16);
    v4f acc[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) acc[kt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const v4f v = tile[col * kLd + 4 * j + quarter];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
          acc[kt] = __builtin_amdgcn_mfma_f32_16x16x4f32(gk[4 * j + e][kt], v[e], acc[kt], 0, 0, 0);
    }
    // acc[kt][r]: basis column 16 kt + 4 quarter + r of pair col
    if (m0 + col < b && 4 * quarter < K) {
      float *dst = dbasis + (int64_t)(m0 + col) * K + 4 * quarter;
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
        __builtin_nontemporal_store(acc[kt], reinterpret_cast<v4f *>(dst + 16 * kt));
    }
  }
}

// ---------------------------------------------------------------------- dfeat ----

constexpr int kMaxRows = 224;         // rows of the LDS table, and less for wide bases, so that two
template <int K>                      // blocks of 64 channels fit a compute unit
constexpr int kRows = K == 64 ? 192 : kMaxRows;
constexpr int kMaxGroup = 64;        // centres per group, one per lane of a wavefront
constexpr int kNoRow = 0xffff;       // pair without a row: added to memory directly
constexpr int kHash = 1024;          // entries of the hash table that numbers the points of a group
constexpr int kProbes = 32;          // places tried for a point before it goes without a row

struct GroupInfo {
  int rows;                          // points of the group that have a row
  int direct;                        // a pair of the group has none
};

// The rows of a group: its points are numbered through a hash table, keys[kMaxRows g ..] are the
// points by number and row_of[m] is the number of pair m.  A pair goes without a row when the
// table is full or when its centre has listed its point before (the products of one centre are
// added without looking at each other).  A kernel of its own, with a small table and so many
// blocks per compute unit: inside the block that multiplies, where the table of sums leaves room
// for two blocks, the chain of dependent loads and probes took 5 of 13 ms.
__global__ void __launch_bounds__(256) group_rows_kernel(
    int64_t n_out, int group, int max_rows, const int2 *__restrict__ nbrs,
    const int *__restrict__ ranges, const int *__restrict__ order,
    unsigned short *__restrict__ row_of, int *__restrict__ keys,
    GroupInfo *__restrict__ info, GroupCentre *__restrict__ listed /* optional */, int64_t pairs,
    int num_basis, float *__restrict__ dbasis) {
  __shared__ int key[kHash];
  __shared__ int number[kHash];
  __shared__ unsigned seen[2][kMaxRows];          // centres of the group that list the row's point
  __shared__ int begin[kMaxGroup], end[kMaxGroup];
  __shared__ int rows, direct;
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int64_t g0 = (int64_t)blockIdx.x * group;
  const int n = (int)(n_out - g0 < group ? n_out - g0 : group);
  if (t < n) {
    const int centre = order[g0 + t];
    begin[t] = centre > 0 ? ranges[centre - 1] : 0;
    end[t] = ranges[centre];
  }
  if (t == 0) rows = direct = 0;
  for (int i = t; i < kHash; i += 256) key[i] = -1;
  for (int i = t; i < kMaxRows; i += 256) seen[0][i] = seen[1][i] = 0;
  __syncthreads();
  for (int i = wave; i < n; i += kWavesPerBlock) {
    for (int m = begin[i] + lane; m < end[i]; m += kWave) {
      const int id = nbrs[m].x;
      int h = (int)(hash_id((unsigned)id) & (kHash - 1));
      for (int probe = 0; probe < kProbes; ++probe) {
        const int got = atomicCAS(&key[h], -1, id);
        if (got == -1 || got == id) break;
        h = (h + 1) & (kHash - 1);
      }
    }
  }
  __syncthreads();
  for (int i = t; i < kHash; i += 256) {
    if (key[i] < 0) continue;
    const int r = atomicAdd(&rows, 1);
    number[i] = r < max_rows ? r : kNoRow;
    if (r < max_rows) keys[(int64_t)blockIdx.x * kMaxRows + r] = key[i];
  }
  __syncthreads();
  for (int i = wave; i < n; i += kWavesPerBlock) {
    for (int m = begin[i] + lane; m < end[i]; m += kWave) {
      const int id = nbrs[m].x;
      int row = kNoRow;
      int h = (int)(hash_id((unsigned)id) & (kHash - 1));
      for (int probe = 0; probe < kProbes; ++probe) {
        if (key[h] == id) {
          row = number[h];
          break;
        }
        h = (h + 1) & (kHash - 1);
      }
      if (row != kNoRow && (atomicOr(&seen[i >> 5][row], 1u << (i & 31)) >> (i & 31)) & 1u)
        row = kNoRow;
      if (row == kNoRow) direct = 1;
      row_of[m] = (unsigned short)row;
    }
  }
  __syncthreads();
  const int used = rows < max_rows ? rows : max_rows;
  if (t == 0) info[blockIdx.x] = GroupInfo{used, direct};
  if (listed && wave == 0) {                      // (n <= 64: a lane each)
    const int count = lane < n ? end[lane] - begin[lane] : 0;
    const unsigned long long any = __ballot(count > 0);
    const int flags = (direct ? 2 : 0) + 4 * used;
    if (count > 0)
      listed[g0 + __popcll(any & ((1ull << lane) - 1ull))] =
          GroupCentre{order[g0 + lane], begin[lane], count, flags + ((any >> lane) == 1 ? 1 : 0)};
    if (any == 0 && lane == 0) listed[g0] = GroupCentre{order[g0], begin[0], 0, flags + 1};
  }
  // rows of the table behind the last centre's pairs (a table of more capacity than pairs)
  for (int64_t i = (int64_t)ranges[n_out - 1] * num_basis + blockIdx.x * 256 + t;
       i < pairs * num_basis; i += (int64_t)gridDim.x * 256)
    dbasis[i] = 0.0f;
}

// W wavefronts of 16 channels each, K basis columns.
template <int W, int K>
struct GroupLds {
  v4f acc[(kRows<K> + 1) * 4 * W];   // sums by row; one more row takes what belongs to no pair
  int key[kMaxRows];
  v4f basis[K == 64 ? 512 : 16 * K]; // basis rows of a chunk
  v4f grad[W][4 * K];                // upstream gradient of its centre, per wavefront
  unsigned short row[64];            // rows of its pairs
  int point[64];                     // and their points, if some pair of the group has no row
};

// Place of 16-byte piece `piece` (of 4 W) in row `row`, in pieces: permuted by the row so that the
// rows a wavefront updates at once fall into different banks.
template <int W>
__device__ __forceinline__ int place(int piece, int row) {
  if constexpr ((W & (W - 1)) == 0) return row * 4 * W + (piece ^ (row & (4 * W - 1)));
  return row * 4 * W + (piece ^ (row & 3));
}

// dfeat^T [c x pair] = G [c x k] B^T [k x pair], one block per (group of centres, part of the
// channels): W wavefronts of 16 channels, kParts blocks for all of them, C <= 16 W kParts
// (kFull: equal).  The pairs of the group are walked centre by centre in chunks of up to 64 (32
// with K = 64).  What a chunk needs -- its basis rows, the rows of its pairs, the upstream
// gradient of its centre -- is fetched two chunks ahead in runs of consecutive lanes and turned
// to operand order in LDS; the wavefronts share the basis rows.  (A row per lane straight into
// the operands costs the address unit four times the cycles and every wavefront its own fetch
// of the basis rows; one chunk ahead leaves 32 KB in flight per compute unit, too few to cover
// the latency of memory.)  A lane ends up with 4 channels of a pair: one 16-byte read, add and
// write of its row in the table.
template <int W, int kParts, int K, bool kFull>
__global__ void __launch_bounds__(64 * W, 2) feature_grads_group_kernel(
    int64_t n_out, int last_pair, int C, int group, const float *__restrict__ basis,
    const int2 *__restrict__ nbrs, const int *__restrict__ ranges, const int *__restrict__ order,
    const unsigned short *__restrict__ row_of, const int *__restrict__ keys,
    const GroupInfo *__restrict__ infos, const float *__restrict__ in_grad,
    float *__restrict__ dfeat) {
  constexpr int kThreads = 64 * W;
  constexpr int kRun = K / 4;                     // basis columns of a quarter
  constexpr int kPieces = K / 4;                  // 16-byte pieces of a basis row
  constexpr int kTiles = K == 64 ? 2 : 4, kChunk = 16 * kTiles;
  constexpr int kFetch = (kChunk * kPieces + kThreads - 1) / kThreads;
  constexpr int kFetchG = (16 * kPieces + 63) / 64;
  constexpr int kNoPair = kRows<K>;               // row of the places behind a centre's last pair
  extern __shared__ __align__(16) char lds_raw[];
  GroupLds<W, K> &s = *reinterpret_cast<GroupLds<W, K> *>(lds_raw);
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int quarter = lane >> 4, col = lane & 15;
  // the parts of a group share its basis rows: numbered onto one XCD (the hardware deals
  // consecutive blocks to the eight XCDs in turn, each with its own L2)
  const int part = (blockIdx.x / 8) % kParts;
  const int64_t which = blockIdx.x / (8 * kParts) * 8 + blockIdx.x % 8, g0 = which * group;
  if (g0 >= n_out) return;
  const GroupInfo info = infos[which];
  const int n = (int)(n_out - g0 < group ? n_out - g0 : group);
  // lane i: centre i of the group, its first pair and their number
  int centres = 0, begins = 0, counts = 0;
  if (lane < n) {
    centres = order[g0 + lane];
    begins = centres > 0 ? ranges[centres - 1] : 0;
    counts = ranges[centres] - begins;
  }
  const unsigned long long listed = __ballot(counts > 0);
  for (int i = t; i < info.rows * 4 * W; i += kThreads) s.acc[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  for (int i = t; i < info.rows; i += kThreads) s.key[i] = keys[which * kMaxRows + i];

  struct Chunk {
    int centre, begin, left, i;                   // left: pairs of the centre from begin on
  };
  auto first_of = [&](int i) {                    // the first chunk of the first centre from i on
    const unsigned long long rest = i < 64 ? listed >> i : 0;
    const int j = i + (rest ? __builtin_ctzll(rest) : 0);
    Chunk c;
    c.i = rest ? j : 64;
    c.centre = __builtin_amdgcn_readlane(centres, j & 63);
    c.begin = __builtin_amdgcn_readlane(begins, j & 63);
    c.left = __builtin_amdgcn_readlane(counts, j & 63);
    return c;
  };
  auto after = [&](const Chunk &c) {
    if (c.left > kChunk) return Chunk{c.centre, c.begin + kChunk, c.left - kChunk, c.i};
    return first_of(c.i + 1);
  };
  const int ch0 = 16 * (part * W + wave);         // the wavefront's first channel
  // (past the last chunk some valid rows are fetched and never used)
  auto fetch = [&](const Chunk &c, v4f (&b)[kFetch], v4f (&g)[kFetchG], int &row, int &point,
                   auto any_direct) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < kFetch; ++x) {
      const int idx = x * kThreads + t, m = c.begin + idx / kPieces;
      b[x] = *reinterpret_cast<const v4f *>(basis + (int64_t)(m < last_pair ? m : last_pair) * K +
                                            4 * (idx % kPieces));
    }
#pragma unroll
    for (int x = 0; x < kFetchG; ++x) {
      const int idx = x * 64 + lane;
      int ch = ch0 + idx / kPieces;
      ch = ch < C ? ch : C - 1;
      g[x] = *reinterpret_cast<const v4f *>(in_grad + ((int64_t)c.centre * C + ch) * K +
                                            4 * (idx % kPieces));
    }
    const int m = c.begin + lane;
    row = row_of[m < last_pair ? m : last_pair];
    if constexpr (any_direct) point = nbrs[m < last_pair ? m : last_pair].x;
    if (lane >= c.left) row = kNoPair;
  };
  auto step = [&](const Chunk &c, const Chunk &ahead, v4f (&b)[kFetch], v4f (&g)[kFetchG],
                  int &row, int &point, auto any_direct) __attribute__((always_inline)) {
    block_lds_sync();                             // the chunk before has been read
#pragma unroll
    for (int x = 0; x < kFetch; ++x) {
      const int idx = x * kThreads + t, slot = idx / kPieces;
      if (kChunk * kPieces % kThreads == 0 || idx < kChunk * kPieces)
        s.basis[slot * kPieces + ((idx % kPieces) ^ (slot & (kPieces - 1)))] = b[x];
    }
#pragma unroll
    for (int x = 0; x < kFetchG; ++x) {
      const int idx = x * 64 + lane, ch = idx / kPieces;
      if (16 * kPieces % 64 == 0 || idx < 16 * kPieces)
        s.grad[wave][ch * kPieces + ((idx % kPieces) ^ (ch & (kPieces - 1)))] = g[x];
    }
    if (wave == 0) {
      s.row[lane] = (unsigned short)row;
      if constexpr (any_direct) s.point[lane] = point;
    }
    block_lds_sync();
    fetch(ahead, b, g, row, point, any_direct);
    auto operand = [&](const v4f *rows, int slot, float (&v)[kRun])
                       __attribute__((always_inline)) {
      if constexpr (kRun >= 4) {
#pragma unroll
        for (int x = 0; x < kRun / 4; ++x) {
          const v4f q = rows[slot * kPieces + ((quarter * (kRun / 4) + x) ^ (slot & (kPieces - 1)))];
#pragma unroll
          for (int e = 0; e < 4; ++e) v[4 * x + e] = q[e];
        }
      } else {
        const float *q = reinterpret_cast<const float *>(
            rows + slot * kPieces + ((quarter >> 1) ^ (slot & (kPieces - 1))));
#pragma unroll
        for (int x = 0; x < kRun; ++x) v[x] = q[(quarter & 1) * kRun + x];
      }
    };
    // The pairs of a centre have distinct rows (or that of no pair): the rows of the chunk are
    // all read before the products and written back after them.
    int at[kTiles];
    bool direct[kTiles];
    float gk[kRun], w[kTiles][kRun];
    v4f have[kTiles], acc[kTiles];
#pragma unroll
    for (int u = 0; u < kTiles; ++u) {
      const int r = s.row[16 * u + col];
      direct[u] = any_direct && r == kNoRow;
      at[u] = place<W>(4 * wave + quarter, direct[u] ? kNoPair : r);
    }
    operand(s.grad[wave], col, gk);
#pragma unroll
    for (int u = 0; u < kTiles; ++u) operand(s.basis, 16 * u + col, w[u]);
#pragma unroll
    for (int u = 0; u < kTiles; ++u) have[u] = s.acc[at[u]];
#pragma unroll
    for (int u = 0; u < kTiles; ++u) acc[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](auto tiles) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < kRun; ++q)
#pragma unroll
        for (int u = 0; u < tiles; ++u)
          acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(gk[q], w[u][q], acc[u], 0, 0, 0);
    };
    // (tiles of 16 without pairs are left out: both gradients of 200 k centres x 36 pairs, 96 x 32 2.52 ->
    // 2.44 ms, 128 x 16 2.10 -> 2.07, 64 x 32 1.60 -> 1.57; 300 k x 50 4.73 -> 4.68, 4.43 -> 4.35, 2.99 ->
    // 2.97; clustered clouds and shorter lists the same as before)
    if (kTiles == 4 && c.left > 48) multiply(std::integral_constant<int, kTiles>{});
    else if (kTiles == 4 && c.left > 32) multiply(std::integral_constant<int, kTiles < 4 ? 2 : 3>{});
    else if (c.left > 16) multiply(std::integral_constant<int, 2>{});
    else multiply(std::integral_constant<int, 1>{});
    // acc[u][r]: channel ch0 + 4 quarter + r of pair 16 u + col
#pragma unroll
    for (int u = 0; u < kTiles; ++u) s.acc[at[u]] = have[u] + acc[u];
    if constexpr (any_direct) {                   // pairs without a row
      const int cc = ch0 + 4 * quarter;
#pragma unroll
      for (int u = 0; u < kTiles; ++u) {
        if (direct[u]) {
          float *dst = dfeat + (int64_t)s.point[16 * u + col] * C + cc;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (kFull || cc + r < C) unsafeAtomicAdd(dst + r, acc[u][r]);
        }
      }
    }
  };
  auto walk = [&](auto any_direct) __attribute__((always_inline)) {
    v4f b0[kFetch], b1[kFetch], g0[kFetchG], g1[kFetchG];
    int row0, row1, point0 = 0, point1 = 0;
    Chunk c = first_of(0), next = after(c);
    fetch(c, b0, g0, row0, point0, any_direct);
    fetch(next, b1, g1, row1, point1, any_direct);
    while (true) {
      if (c.i >= 64) break;
      Chunk ahead = after(next);
      step(c, ahead, b0, g0, row0, point0, any_direct);
      if (next.i >= 64) break;
      c = ahead;
      ahead = after(ahead);
      step(next, ahead, b1, g1, row1, point1, any_direct);
      next = ahead;
    }
  };
  if (info.direct) walk(std::true_type{});
  else walk(std::false_type{});
  __syncthreads();
  // the rows leave: 16 W consecutive floats per row
  for (int i = t; i < info.rows * 16 * W; i += kThreads) {
    const int row = i / (16 * W), c = i - row * (16 * W), dst = 16 * W * part + c;
    if (kFull || dst < C)
      unsafeAtomicAdd(dfeat + (int64_t)s.key[row] * C + dst, s.acc[place<W>(c >> 2, row)][c & 3]);
  }
}

// ----------------------------------------------------------- both gradients at once ----

// For 128 channels and 32 basis columns, where a centre's upstream gradient is 16 KB, one kernel
// forms both gradients.
constexpr int kBothTiles = 8, kBothC = 16 * kBothTiles, kBothK = 32;
constexpr int kBothWaves = 8, kBothThreads = 64 * kBothWaves;
constexpr int kBothChunk = 64;        // pairs of one centre that are worked on at a time
constexpr int kBothRows = 192;        // rows of its table: what 160 KB leave beside a chunk's operands

struct BothLds {
  static constexpr int kLdF = kBothC / 4 + 1;     // 16-byte pieces of a feature row and one of padding
  static constexpr int kLdG = kBothK + 4;         // floats of a channel's upstream gradient, padded
  v4f acc[(kBothRows + 1) * kBothC / 4];          // as in GroupLds
  v4f feat[kBothChunk * kLdF];                    // feature rows of the chunk's pairs
  v4f basis[kBothChunk * kBothK / 4];             // their basis rows
  float grad[kBothC * kLdG];                      // upstream gradient of the centre
  int key[2][kBothRows];                          // points of the group and of the one after
  unsigned short row[kBothChunk];
  int point[kBothChunk];
};
static_assert(sizeof(BothLds) <= 160 * 1024, "one block per compute unit");

// dbasis^T [k x pair] = G^T [k x c] F^T [c x pair] and dfeat^T [c x pair] = G [c x k] B^T [k x pair]
// by one block per compute unit, which walks groups of centres chunk by chunk: the upstream
// gradient, by far the largest operand, comes from memory once for both.  Per chunk the eight
// wavefronts fetch its operands together in runs of consecutive lanes, one chunk ahead and across
// the ends of the groups, and share them through LDS; a wavefront multiplies 16 channels of
// dfeat and a 16 x 16 tile of dbasis.  What is summed in which order is as in the two kernels above.
// 800 k x 52 pairs: 14.2 -> 12.6 ms against the two (2.31 -> 2.08 ms with the numbering of the rows for
// 200 k x 20, 2.50 -> 2.37 for 100 k x 75, clustered clouds of 200 k x 37 3.24 -> 3.13, 100 k x 70 2.35
// both).  Bound by the phases of a chunk one after the other: multiplying 6 ms of it (matrix
// cores 5.3), parking the operands between two barriers 4, and what of the fetch they do
// not cover.  Sixteen wavefronts: 13.0 ms; feature rows from memory straight into the operands and
// two buffers for the rest 13.5; both with 16 basis columns or 64 channels: up to 18 % slower
// than the two kernels, whose upstream gradient is half as large there.  Other shapes have not been
// tried.
__global__ void __launch_bounds__(kBothThreads, 2) both_grads_group_kernel(
    int64_t n_out, int last_pair, int group, int groups, const float *__restrict__ feat,
    const float *__restrict__ basis, const int2 *__restrict__ nbrs,
    const GroupCentre *__restrict__ listed, const unsigned short *__restrict__ row_of,
    const int *__restrict__ keys, const float *__restrict__ in_grad, float *__restrict__ dbasis,
    float *__restrict__ dfeat) {
  constexpr int C = kBothC, K = kBothK;
  constexpr int kRun = K / 4, kPieces = K / 4;
  constexpr int kFetchG = C * kPieces / kBothThreads;
  constexpr int kFetchF = kBothChunk * (C / 4) / kBothThreads;
  constexpr int kNoPair = kBothRows;
  static_assert(kBothChunk * kPieces == kBothThreads, "a piece of the basis rows per thread");
  static_assert(kBothChunk / 16 * (K / 16) == kBothWaves && kBothTiles == kBothWaves &&
                    kRun == kBothTiles, "a tile of either product per wavefront, steps side by side");
  extern __shared__ __align__(16) char lds_raw[];
  BothLds &s = *reinterpret_cast<BothLds *>(lds_raw);
  const int t = threadIdx.x, lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(t / kWave);
  const int quarter = lane >> 4, col = lane & 15;
  const int ch0 = 16 * wave;                                // its channels of dfeat
  const int pair0 = 16 * (wave / 2), k0 = 16 * (wave % 2);  // its pairs and columns of dbasis

  // The reader walks the chunks three ahead of the multiplication.  What it fetches is looked at
  // after the wait for a chunk's operands: a wait of its own would be one for all loads before it,
  // and one for the scalar cache a wait of the LDS accesses.
  using Chunk = GroupChunk;
  const int per_xcd = gridDim.x / 8;              // groups side by side share points: one XCD, one L2
  GroupWalk<kBothChunk> walk(listed, n_out, group, groups, (int)gridDim.x,
                             (int)((blockIdx.x % 8) * per_xcd + blockIdx.x / 8));
  // The point of this lane's pair; past the last one that of the last, since rows behind the lists of
  // a table with spare capacity may hold anything (past the last chunk: of the first row).
  auto point_of = [&](const Chunk &c) {
    const int last = c.left > 0 ? c.left - 1 : 0;
    return nbrs[c.begin + (lane < last ? lane : last)].x;
  };

  v4f fb, fg[kFetchG], ff[kFetchF];
  int frow = kNoPair, fkey = 0, fpoint = 0;
  // (nothing that is fetched is looked at here: the wait for it would be one for every load before)
  auto fetch = [&](const Chunk &c, int ids) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < kFetchF; ++x) {
      const int idx = x * kBothThreads + t;
      ff[x] = *reinterpret_cast<const v4f *>(
          feat + (int64_t)__shfl(ids, idx / (C / 4), kWave) * C + 4 * (idx % (C / 4)));
    }
#pragma unroll
    for (int x = 0; x < kFetchG; ++x)
      fg[x] = __builtin_nontemporal_load(reinterpret_cast<const v4f *>(
          in_grad + (int64_t)c.centre * C * K + 4 * (x * kBothThreads + t)));
    const int m = c.begin + t / kPieces;
    fb = __builtin_nontemporal_load(reinterpret_cast<const v4f *>(
        basis + (int64_t)(m < last_pair ? m : last_pair) * K + 4 * (t % kPieces)));
    if (wave == 0) {
      const int own = c.begin + lane;
      frow = row_of[own < last_pair ? own : last_pair];
      fpoint = ids;
    }
    if (c.first && t < c.rows) fkey = keys[(int64_t)c.group * kMaxRows + t];
  };
  auto park = [&](const Chunk &c) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < kFetchF; ++x) {
      const int idx = x * kBothThreads + t;
      s.feat[idx / (C / 4) * BothLds::kLdF + idx % (C / 4)] = ff[x];
    }
#pragma unroll
    for (int x = 0; x < kFetchG; ++x) {
      const int idx = x * kBothThreads + t;
      *reinterpret_cast<v4f *>(s.grad + idx / kPieces * BothLds::kLdG + 4 * (idx % kPieces)) = fg[x];
    }
    const int slot = t / kPieces;
    s.basis[slot * kPieces + ((t % kPieces) ^ (slot & (kPieces - 1)))] = fb;
    if (wave == 0) {
      s.row[lane] = (unsigned short)(lane < c.left ? frow : kNoPair);
      s.point[lane] = fpoint;
    }
    if (c.first && t < c.rows) s.key[c.odd][t] = fkey;
  };
  // The wavefront's tiles of dfeat go into the table, its tile of dbasis is returned.  With both to
  // multiply it does so in turn: the latter is a chain of dependent instructions.
  auto multiply = [&](const Chunk &c, auto tiles, auto with_basis) __attribute__((always_inline)) {
    constexpr int T = tiles;
    v4f sum = {0.0f, 0.0f, 0.0f, 0.0f};
    int at[T];
    bool direct[T];
    float gk[kRun], w[T][kRun];
    v4f have[T], acc[T];
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int r = s.row[16 * u + col];
      direct[u] = r == kNoRow;
      at[u] = place<kBothTiles>(ch0 / 4 + quarter, direct[u] ? kNoPair : r);
    }
#pragma unroll
    for (int x = 0; x < kRun / 4; ++x) {
      const v4f q = *reinterpret_cast<const v4f *>(s.grad + (ch0 + col) * BothLds::kLdG +
                                                   quarter * kRun + 4 * x);
#pragma unroll
      for (int e = 0; e < 4; ++e) gk[4 * x + e] = q[e];
    }
#pragma unroll
    for (int u = 0; u < T; ++u) {
      const int slot = 16 * u + col;
#pragma unroll
      for (int x = 0; x < kRun / 4; ++x) {
        const v4f q = s.basis[slot * kPieces + ((quarter * (kRun / 4) + x) ^ (slot & (kPieces - 1)))];
#pragma unroll
        for (int e = 0; e < 4; ++e) w[u][4 * x + e] = q[e];
      }
    }
    // The pairs of a centre have distinct rows (or that of no pair): the rows are all read
    // before the products and written back after them.
#pragma unroll
    for (int u = 0; u < T; ++u) {
      have[u] = s.acc[at[u]];
      acc[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int q = 0; q < kRun; ++q) {
#pragma unroll
      for (int u = 0; u < T; ++u)
        acc[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(gk[q], w[u][q], acc[u], 0, 0, 0);
      if constexpr (with_basis) {                 // channels 16 q .. 16 q + 15
        const v4f f = s.feat[(pair0 + col) * BothLds::kLdF + 4 * q + quarter];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          sum = __builtin_amdgcn_mfma_f32_16x16x4f32(
              s.grad[(16 * q + 4 * quarter + e) * BothLds::kLdG + k0 + col], f[e], sum, 0, 0, 0);
      }
    }
#pragma unroll
    for (int u = 0; u < T; ++u) s.acc[at[u]] = have[u] + acc[u];
    if (c.direct) {                               // pairs without a row
#pragma unroll
      for (int u = 0; u < T; ++u) {
        if (!direct[u]) continue;
        float *dst = dfeat + (int64_t)s.point[16 * u + col] * C + ch0 + 4 * quarter;
#pragma unroll
        for (int r = 0; r < 4; ++r) unsafeAtomicAdd(dst + r, acc[u][r]);
      }
    }
    return sum;
  };
  auto products = [&](const Chunk &c) __attribute__((always_inline)) {
    auto by_basis = [&](auto tiles) __attribute__((always_inline)) {
      return pair0 < c.left ? multiply(c, tiles, std::true_type{})
                            : multiply(c, tiles, std::false_type{});
    };
    if (c.left > 48) return by_basis(std::integral_constant<int, 4>{});
    if (c.left > 32) return by_basis(std::integral_constant<int, 3>{});
    if (c.left > 16) return by_basis(std::integral_constant<int, 2>{});
    return by_basis(std::integral_constant<int, 1>{});
  };
  // sum[r]: basis column k0 + 4 quarter + r of pair pair0 + col
  auto store = [&](const Chunk &c, const v4f &sum) __attribute__((always_inline)) {
    if (pair0 + col < c.left)
      __builtin_nontemporal_store(sum, reinterpret_cast<v4f *>(
          dbasis + (int64_t)(c.begin + pair0 + col) * K + k0 + 4 * quarter));
  };
  // the rows leave, consecutive floats each, and the table is empty again
  auto send = [&](const Chunk &c) __attribute__((always_inline)) {
    const int *key = s.key[c.odd];
    for (int i = t; i < c.rows * C; i += kBothThreads) {
      const int row = i / C, ch = i - row * C;
      float &sum = reinterpret_cast<float *>(s.acc + place<kBothTiles>(ch >> 2, row))[ch & 3];
      unsafeAtomicAdd(dfeat + (int64_t)key[row] * C + ch, sum);
      sum = 0.0f;
    }
  };

  for (int i = t; i < kBothRows * C / 4; i += kBothThreads) s.acc[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  walk.fetch();
  Chunk c = walk.read();
  if (c.group < 0) return;
  walk.fetch();
  Chunk next = walk.read();
  walk.fetch();
  Chunk ahead = walk.read();
  walk.fetch();
  fetch(c, point_of(c));
  int ids = point_of(next);
  park(c);
  asm volatile("" : "+v"(ids));                   // (waited for here)
  while (true) {                                  // ends: every step takes a chunk off the list
    block_lds_sync();                             // the chunk is in LDS, the rows before have left
    if (next.group >= 0) {
      fetch(next, ids);
      ids = point_of(ahead);
    }
    const v4f sum = products(c);
    block_lds_sync();                             // the chunk has been read
    // What has been fetched is waited for before anything is written: a wait behind the stores
    // and atomics would be one for them as well.
    if (next.group >= 0) park(next);
    asm volatile("" : "+v"(ids), "+v"(walk.after.centre), "+v"(walk.after.begin),
                 "+v"(walk.after.count), "+v"(walk.after.flags));
    const Chunk third = walk.read();
    walk.fetch();
    store(c, sum);
    if (c.last) send(c);
    if (next.group < 0) break;
    c = next;
    next = ahead;
    ahead = third;
  }
}

// Blocks of 16 channels, or 0 if the shape has no grouped kernel.
static int group_slices(int C, int K) {
  if (K != 8 && K != 16 && K != 32 && K != 64) return 0;
  for (int ct : {1, 2, 4, 6, 8})
    if (C <= 16 * ct) return ct;
  return 0;
}

template <int CT, int K>
static int launch_group(hipStream_t s, int64_t n, int64_t pairs, int C, int group, const float *basis,
                        const float *feat, const int2 *nbrs, const int *ranges, const int *order,
                        const unsigned short *row_of, const int *keys, const GroupInfo *infos,
                        const float *in_grad, float *dbasis, float *dfeat) {
  constexpr int kParts = CT > 4 ? 2 : 1, W = CT / kParts;
  const unsigned grid = (blocks_for(n, group) + 7) / 8 * 8 * kParts;
  const bool full = C == 16 * CT;
  auto dfeat_kernel = full ? feature_grads_group_kernel<W, kParts, K, true>
                           : feature_grads_group_kernel<W, kParts, K, false>;
  MCCNN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(dfeat_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)sizeof(GroupLds<W, K>)));
  hipLaunchKernelGGL(dfeat_kernel, dim3(grid), dim3(64 * W), sizeof(GroupLds<W, K>), s, n,
                     (int)(pairs - 1), C, group,
                     basis, nbrs, ranges, order, row_of, keys, infos, in_grad, dfeat);
  MCCNN_LAUNCH_CHECK();
  auto dbasis_kernel = full ? basis_grads_kernel<CT, K, true> : basis_grads_kernel<CT, K, false>;
  hipLaunchKernelGGL(dbasis_kernel, dim3(wave_grid(n)), dim3(256), 0, s, n, C, feat, nbrs, ranges,
                     order, in_grad, dbasis);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

static int launch_both(hipStream_t s, int64_t n, int64_t pairs, int group, const float *basis,
                       const float *feat, const int2 *nbrs, const GroupCentre *listed,
                       const unsigned short *row_of, const int *keys, const float *in_grad,
                       float *dbasis, float *dfeat) {
  int device = 0, cus = 0;
  MCCNN_HIP_CHECK(hipGetDevice(&device));
  MCCNN_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  // a block per compute unit, in eights (blocks are numbered per XCD)
  const int64_t groups = blocks_for(n, group), wanted = (groups + 7) / 8 * 8;
  const int64_t most = cus < 8 ? 8 : cus / 8 * 8;
  MCCNN_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(both_grads_group_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize,
                                      (int)sizeof(BothLds)));
  hipLaunchKernelGGL(both_grads_group_kernel, dim3((unsigned)(wanted < most ? wanted : most)),
                     dim3(kBothThreads), sizeof(BothLds), s, n, (int)(pairs - 1), group, (int)groups,
                     feat, basis, nbrs, listed, row_of, keys, in_grad, dbasis, dfeat);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

}  // namespace mccnn

using namespace mccnn;

extern "C" size_t mccnn_neighbourhood_order_workspace_bytes(int64_t num_samples) {
  if (num_samples < 0) num_samples = 0;
  return align256(sizeof(unsigned) * (size_t)num_samples) +
         carve_sort_workspace(nullptr, num_samples).bytes;
}

extern "C" int mccnn_neighbourhood_order(mccnn_stream_t stream, int64_t num_samples,
                                         int64_t num_neighbors, const int32_t *neighbors,
                                         const int32_t *ranges, void *workspace,
                                         size_t workspace_bytes, int32_t *order_out) {
  MCCNN_REQUIRE(num_samples >= 0 && num_samples < ((int64_t)1 << 31) && num_neighbors >= 0 &&
                    num_neighbors <= kMostPairs,
                "neighbourhood_order expects fewer than 2^31 centres and at most 2^31 - 1024 pairs");
  if (num_samples == 0) return MCCNN_OK;
  MCCNN_REQUIRE(ranges && workspace && order_out && (neighbors || num_neighbors == 0),
                "neighbourhood_order received a null tensor");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_neighbourhood_order_workspace_bytes(num_samples),
                "neighbourhood_order workspace too small");
  hipStream_t s = as_stream(stream);
  unsigned *keys = (unsigned *)workspace;
  const SortWorkspace w = carve_sort_workspace(
      (char *)workspace + align256(sizeof(unsigned) * (size_t)num_samples), num_samples);
  hipLaunchKernelGGL(neighbourhood_key_kernel, dim3(blocks_for(num_samples * 8, 256)), dim3(256), 0,
                     s, num_samples, (const int2 *)neighbors, ranges, keys);
  MCCNN_LAUNCH_CHECK();
  return sort_order32(s, num_samples, keys, w, order_out);
}

// Where the grouped kernels are the faster ones.  Finding the order takes 0.05 ms (0.17 ms for
// 800 k centres), so a table has to hold work:
// * shapes without a matrix-core kernel with one atomic per pair and channel: from 2^20 pairs x
//   channels on, if the other kernels have as much to do as the order and the groups cost.  Those
//   kernels take about 0.55 ns per pair and 512 elements of C x K (at least one such unit, half
//   as much again at K = 64, and hardly more for many channels at K = 8), plus about 2 us per pair
//   of a centre's serial list; the grouped ones 75 to 125 us up to 200 k pairs, the more the
//   shorter the lists, whose points repeat less.  Other / grouped kernels in us:
//   96 x 8: 4551 centres of 7 pairs 48 / 125, 5461 of 19 130 / 106;
//   24 x 8: 9102 of 7 64 / 122, 36 408 of 7 167 / 150; 64 x 64: 3413 of 7 178 / 144;
//   16 x 8: 13 653 of 7 76 / 119, 109 226 of 7 433 / 186; 3 x 64: 174 762 of 21 3705 / 791.
// * the others: from 2^27 on, and where the atomics are most of the time (many channels or
//   columns) and a group of centres shares its points and fits the table: 16 to 80 pairs per
//   centre (64 x 16 at 30 pairs 2.6 against 2.7 ms).  128 x 32, centres x pairs of uniform and of
//   clustered clouds: 66 k x 17 0.73 / 0.79 and 0.92 / 0.82; 130 k x 18 1.46 / 1.50 and 1.90 / 1.55; 200 k x
//   20 2.43 / 2.20 and 2.99 / 2.30; 100 k x 73 and 47 3.37 / 2.54 and 2.73 / 2.02; 100 k x 88 and 78
//   4.03 / 3.21 and 4.12 / 4.51; 100 k x 115 and 99 5.11 / 6.42 and 5.09 / 6.82.  (Below 16 pairs the
//   line is that of the kernels that form one gradient each, 800 k x 8 7.8 / 8.3; both at once are
//   the faster ones from some 2 M pairs on, 7.8 / 7.5, 400 k x 12 4.16 / 3.85 and 4.50 / 4.04.)
extern "C" int mccnn_basis_proj_grads_grouped_pays(int num_features, int num_basis,
                                                   int64_t num_samples, int64_t num_neighbors) {
  if (group_slices(num_features, num_basis) == 0 || num_samples <= 0 || num_neighbors > kMostPairs)
    return 0;
  const int64_t work = num_neighbors * num_features;
  if (!mfma_grads_supported(num_features, num_basis)) {
    const double units = num_features * num_basis * (num_basis == 64 ? 1.5 : 1.0) / 512;
    const double per_pair = num_basis == 8 ? 0.875 : units > 1 ? units : 1.0;
    return work >= ((int64_t)1 << 20) &&
           num_neighbors * per_pair + 14e3 * num_neighbors / num_samples >= 280e3 ? 1 : 0;
  }
  return work >= ((int64_t)1 << 27) && num_features * num_basis >= 2048 &&
                 num_neighbors >= 16 * num_samples && num_neighbors <= 80 * num_samples
             ? 1 : 0;
}

// Centres per group: about 400 pairs, which list some 140 points where lists overlap as they do in
// space.  Fewer pairs per point than in larger groups, but hardly a group that overflows the
// table's 192 or 224 rows: 800 k x 52 pairs, 128 x 32 take 10.9 / 9.9 / 10.0 / 11.2 ms at 560 /
// 440 / 340 / 240 pairs; both gradients at once (192 rows) 13.8 / 13.3 / 13.2 ms at 460 / 400 / 350,
// clustered clouds of 200 k x 37 3.29 / 3.30 / 3.13.
constexpr double kGroupPairs = 400.0, kBothPairs = 350.0;

// Where both gradients are formed at once.  A block per compute unit walks its share of the groups, and
// with few of them uneven ones do not even out: time of the two kernels over that of the one at
// 1.1 .. 2.2 M pairs of 17 to 57 per centre 0.98 to 1.05 in uniform clouds but 0.94 to 1.00 in
// clustered ones, 2.5 .. 3.2 M 1.02 to 1.04 and 0.97 to 1.01, from 3.9 M on 1.03 to 1.13 and 1.00 to
// 1.07.  (Clustered clouds of more than 64 pairs per centre: 0.95 to 1.03, uniform ones 1.07 to 1.10.)
constexpr int64_t kBothLeast = (int64_t)9 << 18;
static bool both_at_once(int C, int K, int64_t pairs) {
  return C == kBothC && K == kBothK && pairs >= kBothLeast;
}

static int group_centres(int64_t num_samples, int64_t num_neighbors, double pairs) {
  const double mean = (double)num_neighbors / (double)(num_samples > 0 ? num_samples : 1);
  const int group = (int)(pairs / (mean > 1.0 ? mean : 1.0));
  return group < 4 ? 4 : (group > kMaxGroup ? kMaxGroup : group);
}

extern "C" size_t mccnn_basis_proj_grads_grouped_workspace_bytes(int64_t num_samples,
                                                                 int64_t num_neighbors) {
  if (num_samples <= 0 || num_neighbors <= 0) return 0;
  // one size for all shapes: groups as small as any, centres listed where one may have them listed
  const bool both = both_at_once(kBothC, kBothK, num_neighbors);
  const int64_t groups = blocks_for(num_samples, group_centres(num_samples, num_neighbors,
                                                               both ? kBothPairs : kGroupPairs));
  return align256(sizeof(unsigned short) * (size_t)num_neighbors) +
         align256(sizeof(int) * kMaxRows * (size_t)groups) +
         align256(sizeof(GroupInfo) * (size_t)groups) +
         (both ? align256(sizeof(GroupCentre) * (size_t)num_samples) : 0);
}

extern "C" int mccnn_basis_proj_grads_grouped(
    mccnn_stream_t stream, int64_t num_pts, int num_basis, const float *basis, int num_features,
    const float *features, int64_t num_neighbors, const int32_t *neighbors, int64_t num_samples,
    const int32_t *ranges, const int32_t *centre_order, const float *in_grads, void *workspace,
    size_t workspace_bytes, float *basis_grads_out, float *feature_grads_out) {
  const int ct = group_slices(num_features, num_basis);
  MCCNN_REQUIRE(ct > 0,
                "BasisProjGrads (grouped) supports 8/16/32/64 basis functions and at most 128 "
                "features (got %d and %d)", num_basis, num_features);
  MCCNN_REQUIRE(num_pts >= 0 && num_samples >= 0 && num_neighbors >= 0 &&
                    num_neighbors <= kMostPairs && num_samples < ((int64_t)1 << 31),
                "BasisProjGrads (grouped) expects fewer than 2^31 centres and at most 2^31 - 1024 "
                "pairs");
  hipStream_t s = as_stream(stream);
  if (num_pts > 0) {
    MCCNN_REQUIRE(feature_grads_out, "BasisProjGrads (grouped) received a null tensor");
    int rc = fill_zero(s, feature_grads_out, sizeof(float) * (size_t)num_pts * num_features);
    if (rc != MCCNN_OK) return rc;
  }
  if (num_samples == 0 || num_neighbors == 0) return MCCNN_OK;
  MCCNN_REQUIRE(ranges && centre_order && basis && features && neighbors && in_grads &&
                    basis_grads_out,
                "BasisProjGrads (grouped) received a null tensor");
  MCCNN_REQUIRE(workspace && workspace_bytes >= mccnn_basis_proj_grads_grouped_workspace_bytes(
                                                     num_samples, num_neighbors),
                "BasisProjGrads (grouped) workspace too small");
  const bool both = both_at_once(num_features, num_basis, num_neighbors);
  const int group = group_centres(num_samples, num_neighbors, both ? kBothPairs : kGroupPairs);
  const int64_t groups = blocks_for(num_samples, group);
  unsigned short *row_of = (unsigned short *)workspace;
  int *keys = (int *)((char *)workspace + align256(sizeof(unsigned short) * (size_t)num_neighbors));
  GroupInfo *infos = (GroupInfo *)((char *)keys + align256(sizeof(int) * kMaxRows * (size_t)groups));
  GroupCentre *listed =
      both ? (GroupCentre *)((char *)infos + align256(sizeof(GroupInfo) * (size_t)groups)) : nullptr;
  hipLaunchKernelGGL(group_rows_kernel, dim3((unsigned)groups), dim3(256), 0, s, num_samples, group,
                     both ? kBothRows : num_basis == 64 ? kRows<64> : kMaxRows,
                     (const int2 *)neighbors, ranges, centre_order, row_of, keys, infos,
                     listed, num_neighbors, num_basis, basis_grads_out);
  MCCNN_LAUNCH_CHECK();
  int rc = MCCNN_OK;
  if (both)
    return launch_both(s, num_samples, num_neighbors, group, basis, features,
                       (const int2 *)neighbors, listed, row_of, keys, in_grads, basis_grads_out,
                       feature_grads_out);
#define MCCNN_GROUP_K(CT_, K_)                                                                   \
  rc = launch_group<CT_, K_>(s, num_samples, num_neighbors, num_features, group, basis, features, \
                             (const int2 *)neighbors, ranges, centre_order, row_of, keys, infos, \
                             in_grads,                                                           \
                             basis_grads_out, feature_grads_out)
#define MCCNN_GROUP(CT_)                         \
  switch (num_basis) {                           \
    case 8: MCCNN_GROUP_K(CT_, 8); break;        \
    case 16: MCCNN_GROUP_K(CT_, 16); break;      \
    case 32: MCCNN_GROUP_K(CT_, 32); break;      \
    default: MCCNN_GROUP_K(CT_, 64); break;      \
  }
  switch (ct) {
    case 1: MCCNN_GROUP(1); break;
    case 2: MCCNN_GROUP(2); break;
    case 4: MCCNN_GROUP(4); break;
    case 6: MCCNN_GROUP(6); break;
    default: MCCNN_GROUP(8); break;
  }
#undef MCCNN_GROUP
#undef MCCNN_GROUP_K
  return rc;
}
