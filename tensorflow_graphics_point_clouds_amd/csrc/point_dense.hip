// Gradients of the feature-space layers between the point convolutions: batch normalisation over
// the points with the leaky activation behind it, and the per-point linear map
// (pylib/pc/layers/Conv1x1.py:24-101, pylib/pc/layers/network_blocks.py:27-465, the
// BatchNormalization and LeakyReLU layers of modelnet40.py:128-260).  No counterpart among the
// reference's ops (TensorFlow's own kernels).
//
// A level of a network holds a thousand to some ten thousand points with 16 to 256 features:
// 0.1 to 16 MB, microseconds at the rate of memory, so what counts is the number of launches and
// what the host does for each.  Normalisation + activation take two launches (column sums per
// slab of points; then every block adds the partial sums of its columns up by itself and maps
// its points), against three of the separate torch operations; the linear map takes one for its
// input and two for weights and bias.
// The forward passes stay torch's own kernels: which side of 0 a point lies on is decided there,
// and a network's gradients jump where another rounding moves a point across.
//
// Forward + backward through autograd, before -> with these kernels (torch's forward in both):
// normalisation + activation of 100 k x 256 849 -> 520 us, 16 k x 256 173 -> 119 us; linear
// 1200 x 64 -> 64 129 -> 95 us (the host's time), 100 k x 64 -> 64 375 -> 96 us, 800 k x 64 -> 64
// 1.90 -> 0.47 ms (torch sums the weight gradient over all points in few blocks).
#include "common.h"
#include "mfma.h"

namespace mccnn {

// ------------------------------------------------------------ normalisation + activation ----

// A block has kLanes lanes of four columns (16 or, up to 16 columns, 4) and 256 / kLanes points
// per step.
constexpr int kMaxSlabs = 256;
constexpr int kMapRows = 512;        // points of a block that maps them, at most

// Points per slab: every block that maps points reads all partial sums of its columns, so there
// are at most 64 slabs up to 16 k points (64 to 256 points each) and 256 above, where a pass
// over the points is long enough to hide them.
static int64_t norm_slab_rows(int64_t n) {
  const int64_t slabs = n <= 16384 ? 64 : kMaxSlabs, least = n <= 16384 ? 64 : 256;
  const int64_t rows = (n + slabs - 1) / slabs;
  return ((rows < least ? least : rows) + 63) / 64 * 64;
}

template <bool kVec>
__device__ __forceinline__ v4f load_cols(const float *__restrict__ p, int c, int C) {
  if (kVec) return *reinterpret_cast<const v4f *>(p + c);
  v4f v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = c + e < C ? p[c + e] : 0.0f;
  return v;
}

template <bool kVec>
__device__ __forceinline__ void store_cols(float *__restrict__ p, int c, int C, const v4f &v) {
  if (kVec) {
    *reinterpret_cast<v4f *>(p + c) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < C) p[c + e] = v[e];
  }
}

// The sum over the points of a block's step, of two values per column; partial is [slab][2][C].
template <int kLanes>
__device__ __forceinline__ void store_partials(v4f a, v4f b, int slab, int c, int C,
                                               float *__restrict__ partial) {
  constexpr int kRows = 256 / kLanes;
  __shared__ v4f parts[2][kRows][kLanes];
  const int lane = threadIdx.x % kLanes, row = threadIdx.x / kLanes;
  parts[0][row][lane] = a;
  parts[1][row][lane] = b;
  __syncthreads();
  if (threadIdx.x < 2 * kLanes) {
    v4f sum = parts[row][0][lane];               // row: which of the two
#pragma unroll
    for (int r = 1; r < kRows; ++r) sum += parts[row][r][lane];
    float *out = partial + ((int64_t)slab * 2 + row) * C;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (c + e < C) out[c + e] = sum[e];
  }
}

// Adds the partial sums of the block's columns up (in double: sums over all points) into
// sums[2][4 kLanes]; every thread of the block.
template <int kLanes>
__device__ __forceinline__ void gather_partials(const float *__restrict__ partial, int slabs, int C,
                                                double (*sums)[4 * kLanes]) {
  constexpr int kCols = 4 * kLanes, kParts = 256 / (2 * kCols);
  __shared__ double parts[kParts][2][kCols];
  const int col = threadIdx.x % kCols, which = threadIdx.x / kCols % 2,
            first = threadIdx.x / (2 * kCols);
  const int c = blockIdx.y * kCols + col;
  double sum = 0.0;
  if (c < C)
    for (int s = first; s < slabs; s += kParts)
      sum += (double)partial[((int64_t)s * 2 + which) * C + c];
  parts[first][which][col] = sum;
  __syncthreads();
  if (first == 0) {
#pragma unroll
    for (int i = 1; i < kParts; ++i) sum += parts[i][which][col];
    sums[which][col] = sum;
  }
  __syncthreads();
}

struct NormArgs {
  const float *x, *y, *g;            // input, output (after the activation), its gradient [n, C]
  const float *mean, *inv, *weight;  // statistics of the forward pass, scale [C]
  float slope;
};

// The parameters of a lane's four columns.
struct NormCols {
  v4f mean, inv, weight;
};

template <bool kVec>
__device__ __forceinline__ NormCols norm_cols(const NormArgs &a, int c, int C) {
  return NormCols{load_cols<kVec>(a.mean, c, C), load_cols<kVec>(a.inv, c, C),
                  load_cols<kVec>(a.weight, c, C)};
}

// dz = g act'(z) of a point's four columns, xhat = (x - mean) inv beside it.  The activation
// keeps signs, so that its result tells on which side of 0 the forward pass saw z.  NaN takes the
// side that torch's activations give it: ReLU passes its gradient, a slope applies.
template <bool kVec>
__device__ __forceinline__ v4f norm_dz(const NormArgs &a, int64_t i, int c, int C,
                                       const NormCols &p, v4f *xhat) {
  *xhat = (load_cols<kVec>(a.x + i * C, c, C) - p.mean) * p.inv;
  v4f dz = load_cols<kVec>(a.g + i * C, c, C);
  if (a.slope != 1.0f) {
    const v4f y = load_cols<kVec>(a.y + i * C, c, C);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (a.slope == 0.0f) dz[e] = y[e] <= 0.0f ? 0.0f : dz[e];
      else if (!(y[e] > 0.0f)) dz[e] = a.slope * dz[e];
  }
  return dz;
}

template <int kLanes, bool kVec>
__global__ void __launch_bounds__(256) norm_grad_sums_kernel(int64_t n, int C, int64_t slab_rows,
                                                             NormArgs a,
                                                             float *__restrict__ partial) {
  const int c = 4 * (blockIdx.y * kLanes + threadIdx.x % kLanes);
  const int64_t first = (int64_t)blockIdx.x * slab_rows;
  const int64_t last = first + slab_rows < n ? first + slab_rows : n;
  v4f s1 = {0.0f, 0.0f, 0.0f, 0.0f}, s2 = s1;
  if (c < C) {
    const NormCols p = norm_cols<kVec>(a, c, C);
#pragma unroll 2
    for (int64_t i = first + threadIdx.x / kLanes; i < last; i += 256 / kLanes) {
      v4f xhat;
      const v4f dz = norm_dz<kVec>(a, i, c, C, p, &xhat);
      s1 += dz;
      s2 += dz * xhat;
    }
  }
  store_partials<kLanes>(s1, s2, blockIdx.x, c, C, partial);
}

// dx = w inv (dz - mean(dz) - xhat mean(dz xhat)), or w inv dz when the statistics were given
// (`fixed`); dweight = sum dz xhat, dbias = sum dz.
template <int kLanes, bool kVec>
__global__ void __launch_bounds__(256) norm_grads_kernel(
    int64_t n, int C, int64_t map_rows, int slabs, NormArgs a, int fixed,
    const float *__restrict__ partial, float *__restrict__ dx, float *__restrict__ dweight,
    float *__restrict__ dbias) {
  __shared__ double sums[2][4 * kLanes];
  __shared__ float means[2][4 * kLanes];
  gather_partials<kLanes>(partial, slabs, C, sums);
  if (threadIdx.x < 4 * kLanes) {
    const int col = threadIdx.x, c = blockIdx.y * 4 * kLanes + col;
    means[0][col] = fixed ? 0.0f : (float)(sums[0][col] / (double)n);
    means[1][col] = fixed ? 0.0f : (float)(sums[1][col] / (double)n);
    if (blockIdx.x == 0 && c < C) {
      dbias[c] = (float)sums[0][col];
      dweight[c] = (float)sums[1][col];
    }
  }
  __syncthreads();
  const int lane = threadIdx.x % kLanes, c = 4 * (blockIdx.y * kLanes + lane);
  if (c >= C || dx == nullptr) return;
  const NormCols p = norm_cols<kVec>(a, c, C);
  const v4f m1 = *reinterpret_cast<const v4f *>(means[0] + 4 * lane);
  const v4f m2 = *reinterpret_cast<const v4f *>(means[1] + 4 * lane);
  const int64_t first = (int64_t)blockIdx.x * map_rows;
  const int64_t last = first + map_rows < n ? first + map_rows : n;
  for (int64_t i = first + threadIdx.x / kLanes; i < last; i += 256 / kLanes) {
    v4f xhat;
    const v4f dz = norm_dz<kVec>(a, i, c, C, p, &xhat);
    // (with given statistics an infinite point has a finite gradient)
    store_cols<kVec>(dx + i * C, c, C, (fixed ? dz : dz - m1 - xhat * m2) * (p.inv * p.weight));
  }
}

// ------------------------------------------------------------------- linear map ----

constexpr int kLinRows = 32, kLinCols = 64;     // output tile of a block
constexpr int kLinDepth = 32;                   // reduction per step
constexpr int kLinLd = kLinDepth + 4;

// out [n, F] = x [n, R] w^T for w [F, R].  Blocks of four wavefronts with 16 x 32 outputs each,
// tiles small enough that a few thousand points fill the device; the operands of the next step
// are in flight during a step.  In LDS the reduction runs along the rows of both, so that a lane
// reads four of its terms (16 j + 4 quarter + e) at once.
template <bool kVec>
__global__ void __launch_bounds__(256) linear_input_grads_kernel(int64_t n, int R, int F,
                                                                 const float *__restrict__ x,
                                                                 const float *__restrict__ w,
                                                                 float *__restrict__ out) {
  __shared__ __align__(16) float xs[kLinRows][kLinLd];
  __shared__ __align__(16) float ws[kLinCols][kLinLd];
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int quarter = lane >> 4, col = lane & 15;
  const int64_t row0 = (int64_t)blockIdx.x * kLinRows;
  const int f0 = blockIdx.y * kLinCols;
  v4f nx, nw[2];
  auto fetch = [&](int k0) __attribute__((always_inline)) {
    {                                              // x: 8 pieces per row
      const int64_t i = row0 + t / 8;
      const int k = k0 + 4 * (t % 8);
      nx = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      if (i < n && k < R) nx = load_cols<kVec>(x + i * R, k, R);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      nw[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      const int f = f0 + t / 8 + 32 * j, k = k0 + 4 * (t % 8);
      if (f < F && k < R) nw[j] = load_cols<kVec>(w + (int64_t)f * R, k, R);
    }
  };
  v4f acc[2];
  acc[0] = acc[1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  const int wr = 16 * (wave & 1), wc = 32 * (wave >> 1);
  fetch(0);
  for (int k0 = 0; k0 < R; k0 += kLinDepth) {
    __syncthreads();
    *reinterpret_cast<v4f *>(&xs[t / 8][4 * (t % 8)]) = nx;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<v4f *>(&ws[t / 8 + 32 * j][4 * (t % 8)]) = nw[j];
    __syncthreads();
    if (k0 + kLinDepth < R) fetch(k0 + kLinDepth);
#pragma unroll
    for (int j = 0; j < kLinDepth / 16; ++j) {
      const int k = 16 * j + 4 * quarter;
      const v4f a = *reinterpret_cast<const v4f *>(&xs[wr + col][k]);
      const v4f b0 = *reinterpret_cast<const v4f *>(&ws[wc + col][k]);
      const v4f b1 = *reinterpret_cast<const v4f *>(&ws[wc + 16 + col][k]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b0[e], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b1[e], acc[1], 0, 0, 0);
      }
    }
  }
  // acc[u][r]: row wr + 4 quarter + r, column wc + 16 u + col
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int f = f0 + wc + 16 * u + col;
    if (f >= F) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t i = row0 + wr + 4 * quarter + r;
      if (i < n) out[i * F + f] = acc[u][r];
    }
  }
}

constexpr int kTile = 64;                         // output tile of the weight gradient
constexpr int kStep = 32;                         // points per step

static int64_t linear_slabs(int64_t n, int R, int F) {
  const int64_t tiles = (int64_t)((R + kTile - 1) / kTile) * ((F + kTile - 1) / kTile);
  // At least four steps each and enough blocks to fill the device; a serial sum over more than
  // 2048 points would cost accuracy (1e-6 of the result at 12 500 points per slab).
  const int64_t most = tiles >= 8 ? 32 : 256 / tiles, wanted = (n + 127) / 128,
                least = (n + 2047) / 2048;
  const int64_t slabs = wanted > most ? most : wanted;
  return slabs > least ? slabs : least;
}

// Per slab of points, dw [R, F] = x^T g and db [F] = sum of g; partial [slab][R F + F].
template <bool kVecX, bool kVecG>
__global__ void __launch_bounds__(256) linear_weight_grads_kernel(
    int64_t n, int R, int F, int64_t slab_rows, const float *__restrict__ x,
    const float *__restrict__ g, float *__restrict__ partial) {
  __shared__ __align__(16) float xs[kStep][kTile + 4];
  __shared__ __align__(16) float gs[kStep][kTile + 4];
  __shared__ v4f sums[16][16];
  const int t = threadIdx.x, lane = lane_id(), wave = t / kWave;
  const int quarter = lane >> 4, col = lane & 15;
  const int r0 = blockIdx.z * kTile, f0 = blockIdx.y * kTile;
  const int64_t first = (int64_t)blockIdx.x * slab_rows;
  const int64_t last = first + slab_rows < n ? first + slab_rows : n;
  v4f nx[2], ng[2], bias = {0.0f, 0.0f, 0.0f, 0.0f};
  auto fetch = [&](int64_t i0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int64_t i = i0 + t / 16 + 16 * j;
      const int c = 4 * (t % 16);
      nx[j] = ng[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      if (i < last) {
        if (r0 + c < R) nx[j] = load_cols<kVecX>(x + i * R, r0 + c, R);
        if (f0 + c < F) ng[j] = load_cols<kVecG>(g + i * F, f0 + c, F);
      }
    }
  };
  v4f acc[2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u) acc[u][0] = acc[u][1] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  const int wr = 32 * (wave & 1), wc = 32 * (wave >> 1);
  fetch(first);
  for (int64_t i0 = first; i0 < last; i0 += kStep) {
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      *reinterpret_cast<v4f *>(&xs[t / 16 + 16 * j][4 * (t % 16)]) = nx[j];
      *reinterpret_cast<v4f *>(&gs[t / 16 + 16 * j][4 * (t % 16)]) = ng[j];
      bias += ng[j];
    }
    __syncthreads();
    if (i0 + kStep < last) fetch(i0 + kStep);
#pragma unroll
    for (int k = 0; k < kStep; k += 4) {
      float a[2], b[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        a[u] = xs[k + quarter][wr + 16 * u + col];
        b[u] = gs[k + quarter][wc + 16 * u + col];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
          acc[u][v] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[u], b[v], acc[u][v], 0, 0, 0);
    }
  }
  float *out = partial + (int64_t)blockIdx.x * ((int64_t)R * F + F);
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int i = r0 + wr + 16 * u + 4 * quarter + r, f = f0 + wc + 16 * v + col;
        if (i < R && f < F) out[(int64_t)i * F + f] = acc[u][v][r];
      }
  if (blockIdx.z == 0) {
    sums[t / 16][t % 16] = bias;
    __syncthreads();
    if (t < 16) {
      v4f sum = sums[0][t];
#pragma unroll
      for (int r = 1; r < 16; ++r) sum += sums[r][t];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (f0 + 4 * t + e < F) out[(int64_t)R * F + f0 + 4 * t + e] = sum[e];
    }
  }
}

// The slabs' parts added in their order.
__global__ void __launch_bounds__(256) linear_reduce_kernel(int64_t count, int64_t weights,
                                                            int slabs,
                                                            const float *__restrict__ partial,
                                                            float *__restrict__ dw,
                                                            float *__restrict__ db) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float sum = 0.0f;
#pragma unroll 8
  for (int s = 0; s < slabs; ++s) sum += partial[s * count + i];
  if (i < weights) dw[i] = sum;
  else if (db) db[i - weights] = sum;
}

}  // namespace mccnn

using namespace mccnn;

#define MCCNN_BOOL_SWITCH(cond_, name_, ...)                     \
  if (cond_) { constexpr bool name_ = true; __VA_ARGS__; }       \
  else { constexpr bool name_ = false; __VA_ARGS__; }

static bool aligned16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

extern "C" size_t mccnn_norm_act_grads_workspace_bytes(int num_features) {
  return num_features > 0 ? sizeof(float) * 2 * kMaxSlabs * (size_t)num_features : 0;
}

extern "C" int mccnn_norm_act_grads(mccnn_stream_t stream, int64_t num_pts, int num_features,
                                    const float *x, const float *y, const float *in_grads,
                                    const float *mean, const float *inv_std, const float *weight,
                                    int training, float slope, void *workspace,
                                    size_t workspace_bytes, float *x_grads_out,
                                    float *weight_grads_out, float *bias_grads_out) {
  MCCNN_REQUIRE(num_pts > 0 && num_features > 0 && num_features <= 65535 * 64,
                "NormActGrads expects points and features");
  MCCNN_REQUIRE(slope >= 0.0f, "NormActGrads expects a slope of at least 0 (got %g)", slope);
  MCCNN_REQUIRE(x && y && in_grads && mean && inv_std && weight && workspace && weight_grads_out &&
                    bias_grads_out,
                "NormActGrads received a null tensor");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_norm_act_grads_workspace_bytes(num_features),
                "NormActGrads workspace too small");
  hipStream_t s = as_stream(stream);
  const NormArgs a{x, y, in_grads, mean, inv_std, weight, slope};
  const int64_t rows = norm_slab_rows(num_pts), map_rows = rows < kMapRows ? rows : kMapRows;
  const int slabs = (int)blocks_for(num_pts, rows), tiles = (num_features + 63) / 64;
  const dim3 grid(slabs, tiles), map_grid(blocks_for(num_pts, map_rows), tiles), block(256);
  float *partial = (float *)workspace;
  bool vec = num_features % 4 == 0;
  for (const void *p : {(const void *)x, (const void *)y, (const void *)in_grads,
                        (const void *)mean, (const void *)inv_std, (const void *)weight,
                        (const void *)x_grads_out})
    vec = vec && aligned16(p);
  MCCNN_BOOL_SWITCH(vec, kVec, MCCNN_BOOL_SWITCH(num_features <= 16, kNarrow, {
    constexpr int kLanes = kNarrow ? 4 : 16;
    hipLaunchKernelGGL((norm_grad_sums_kernel<kLanes, kVec>), grid, block, 0, s, num_pts,
                       num_features, rows, a, partial);
    MCCNN_LAUNCH_CHECK();
    hipLaunchKernelGGL((norm_grads_kernel<kLanes, kVec>), map_grid, block, 0, s, num_pts,
                       num_features, map_rows, slabs, a, training ? 0 : 1, partial, x_grads_out,
                       weight_grads_out, bias_grads_out);
  }));
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

static int check_linear(const char *op, int64_t num_rows, int cols_in, int cols_out) {
  MCCNN_REQUIRE(num_rows >= 0 && num_rows <= ((int64_t)1 << 31) - kLinRows && cols_in > 0 &&
                    cols_out > 0 && cols_in <= 65536 && cols_out <= 65536,
                "%s expects up to 2^31 rows and 1 to 65536 columns", op);
  return MCCNN_OK;
}

extern "C" int mccnn_linear_input_grads(mccnn_stream_t stream, int64_t num_rows, int num_cols_in,
                                        const float *weights, int num_cols_out,
                                        const float *in_grads, float *x_grads_out) {
  int rc = check_linear("LinearInputGrads", num_rows, num_cols_in, num_cols_out);
  if (rc != MCCNN_OK || num_rows == 0) return rc;
  MCCNN_REQUIRE(weights && in_grads && x_grads_out, "LinearInputGrads received a null tensor");
  const dim3 grid(blocks_for(num_rows, kLinRows), (num_cols_in + kLinCols - 1) / kLinCols);
  const bool vec = num_cols_out % 4 == 0 && aligned16(in_grads) && aligned16(weights);
  MCCNN_BOOL_SWITCH(vec, kVec, {
    hipLaunchKernelGGL(linear_input_grads_kernel<kVec>, grid, dim3(256), 0, as_stream(stream),
                       num_rows, num_cols_out, num_cols_in, in_grads, weights, x_grads_out);
  });
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" size_t mccnn_linear_weight_grads_workspace_bytes(int64_t num_rows, int num_cols_in,
                                                            int num_cols_out) {
  if (num_rows <= 0 || num_cols_in <= 0 || num_cols_out <= 0) return 0;
  return sizeof(float) * (size_t)linear_slabs(num_rows, num_cols_in, num_cols_out) *
         ((size_t)num_cols_in * num_cols_out + num_cols_out);
}

extern "C" int mccnn_linear_weight_grads(mccnn_stream_t stream, int64_t num_rows, int num_cols_in,
                                         const float *x, int num_cols_out, const float *in_grads,
                                         void *workspace, size_t workspace_bytes,
                                         float *weight_grads_out, float *bias_grads_out) {
  int rc = check_linear("LinearWeightGrads", num_rows, num_cols_in, num_cols_out);
  if (rc != MCCNN_OK) return rc;
  MCCNN_REQUIRE(num_rows > 0 && x && in_grads && workspace && weight_grads_out,
                "LinearWeightGrads received a null tensor");
  MCCNN_REQUIRE(workspace_bytes >= mccnn_linear_weight_grads_workspace_bytes(num_rows, num_cols_in,
                                                                             num_cols_out),
                "LinearWeightGrads workspace too small");
  hipStream_t s = as_stream(stream);
  int64_t slabs = linear_slabs(num_rows, num_cols_in, num_cols_out);
  const int64_t rows = ((num_rows + slabs - 1) / slabs + kStep - 1) / kStep * kStep;
  slabs = (num_rows + rows - 1) / rows;
  const dim3 grid((unsigned)slabs, (num_cols_out + kTile - 1) / kTile,
                  (num_cols_in + kTile - 1) / kTile);
  const bool vx = num_cols_in % 4 == 0 && aligned16(x);
  const bool vg = num_cols_out % 4 == 0 && aligned16(in_grads);
  MCCNN_BOOL_SWITCH(vx, kVx, MCCNN_BOOL_SWITCH(vg, kVg, {
    hipLaunchKernelGGL((linear_weight_grads_kernel<kVx, kVg>), grid, dim3(256), 0, s, num_rows,
                       num_cols_in, num_cols_out, rows, x, in_grads, (float *)workspace);
  }));
  MCCNN_LAUNCH_CHECK();
  const int64_t weights = (int64_t)num_cols_in * num_cols_out, count = weights + num_cols_out;
  hipLaunchKernelGGL(linear_reduce_kernel, dim3(blocks_for(count, 256)), dim3(256), 0, s, count,
                     weights, (int)slabs, (const float *)workspace, weight_grads_out,
                     bias_grads_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}
