// Feature gradient of a convolution layer with few input channels (MCConv.py:137-194,
// KPConv.py:165-232), from the gradient of its projection:
//     dfeat[j, c] = sum over the pairs (i, j) of sum_k basis_k(ij) G[i, c, k],
//     G = dout W^T as [N_out, C, 16].
// The transposed convolution (mc_conv.hip run backwards) gathers the F output columns of a
// centre per pair and leaves an [N, F, 16] tensor for the product with the weights; here a pair
// gathers the 16 C values of its centre's G, and the sums over pairs and basis columns end in the
// C channels at once.  With C <= 16 and F larger the rows are as long or little longer, nothing
// of F columns reaches memory, and every value is multiplied once in vector instructions where the
// matrix cores would have to multiply F of them.
//
// A wavefront takes a run of consecutive points, whose pairs (of the transposed table) are one
// stretch, and stages 64 of them at a time in LDS as the projection does (offset, weight, row of
// G); the indices and coordinates of the next 64 are in flight meanwhile.  A quarter of the
// wavefront takes a pair: lane `col` evaluates basis column col of it, reads G[., c, col] of every
// channel (16 lanes: 64 contiguous bytes) and keeps a sum per channel.  At a point's end the
// 64 x C partial sums are folded by exchanges that halve the values a lane holds.
#include "common.h"
#include "mfma.h"
#include "mc_conv.h"

namespace mccnn {

constexpr int kGatherRun = 8;      // points per wavefront, at most
constexpr int kGatherAhead = 2;    // pairs of a quarter in flight

// kLive: channels that are gathered, of rows of G of `row_bytes`; columns c < live of `out` are
// written.  kWhole: a row holds kLive channels or more.  Where it holds fewer the last one is read
// again in their place (nothing behind the row, or behind G, is).
template <int kLive, int D, bool kWhole, class Basis>
__device__ __forceinline__ void gather_grads_body(
    int64_t n_pts, int run_len, const char *__restrict__ grads, unsigned row_bytes,
    const int2 *__restrict__ nbrs, const int *__restrict__ ranges, const McParams<D> &p,
    const Basis &basis, const int *__restrict__ out_rows, int live, bool add,
    float *__restrict__ out, PairStage *stage) {
  const int lane = lane_id();
  const int64_t c0 = wave_slot_xcd() * run_len;
  if (c0 >= n_pts) return;
  const int nc = (int)(n_pts - c0 < run_len ? n_pts - c0 : run_len);
  const int quarter = lane >> 4, col = lane & 15;
  int my_end = 0, my_row = 0;             // lane i < nc: end offset and output row of point c0 + i
  if (lane < nc) {
    my_end = ranges[c0 + lane];
    my_row = out_rows ? out_rows[c0 + lane] : (int)(c0 + lane);
  }
  const int begin = c0 > 0 ? ranges[c0 - 1] : 0;
  int ends[kGatherRun];
#pragma unroll
  for (int i = 0; i < kGatherRun; ++i)
    ends[i] = __builtin_amdgcn_readlane(my_end, i < nc ? i : nc - 1);
  const int total_end = ends[kGatherRun - 1];
  float ir[D];
#pragma unroll
  for (int d = 0; d < D; ++d) ir[d] = p.inv_radii[d];
  const unsigned last_channel = row_bytes - 64;

  struct Pending {
    int idx;
    float ctr[D], pt[D], pdf;
  };
  auto fetch_index = [&](int m0) { return m0 + lane < total_end ? nbrs[m0 + lane].x : 0; };
  auto fetch_rest = [&](int m0, int idx) {
    Pending q;
    q.idx = idx;
    q.pdf = 1.0f;
#pragma unroll
    for (int d = 0; d < D; ++d) q.ctr[d] = q.pt[d] = 0.0f;
    const int m = m0 + lane;
    if (m < total_end) {
      int ci = 0;                         // point of pair m inside the run
#pragma unroll
      for (int i = 0; i < kGatherRun - 1; ++i) ci += m >= ends[i] ? 1 : 0;
#pragma unroll
      for (int d = 0; d < D; ++d) {
        q.ctr[d] = p.pout[(c0 + ci) * D + d];
        q.pt[d] = p.pin[(int64_t)idx * D + d];
      }
      if (p.pdf) q.pdf = p.pdf[m];
    }
    return q;
  };

  float acc[kLive];
#pragma unroll
  for (int c = 0; c < kLive; ++c) acc[c] = 0.0f;
  auto finish_point = [&](int i) {        // fold, store and clear the sums of point c0 + i
    float v[kLive];
#pragma unroll
    for (int c = 0; c < kLive; ++c) {
      v[c] = acc[c];
      acc[c] = 0.0f;
    }
    int channel = 0;
#pragma unroll
    for (int off = 1, left = kLive; off < kWave; off <<= 1) {
      if (left > 1) {
        left >>= 1;
        const bool high = lane & off;
#pragma unroll
        for (int c = 0; c < left; ++c) {
          const float keep = high ? v[c + left] : v[c], send = high ? v[c] : v[c + left];
          v[c] = keep + __shfl_xor(send, off, kWave);
        }
        channel += high ? left : 0;
      } else {
        v[0] += __shfl_xor(v[0], off, kWave);
      }
    }
    const int64_t row = __builtin_amdgcn_readlane(my_row, i);
    if (lane < kLive && channel < live) {
      float *o = out + row * live + channel;
      *o = add ? *o + v[0] : v[0];
    }
  };

  int cur = 0, cur_start = begin, cur_end = ends[0];
  Pending pend = fetch_rest(begin, fetch_index(begin));
  int next_idx = fetch_index(begin + kWave);
  for (int m0 = begin; m0 < total_end; m0 += kWave) {
    const int cnt = total_end - m0 < kWave ? total_end - m0 : kWave;
    float dl[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < D; ++d) dl[d] = (pend.pt[d] - pend.ctr[d]) * ir[d];
    wave_lds_sync();                      // the previous chunk has been read
    stage->geo[lane] = make_float4(dl[0], dl[1], dl[2], 1.0f / pend.pdf);
    stage->row[lane] = (unsigned)pend.idx * row_bytes;
    wave_lds_sync();
    pend = fetch_rest(m0 + kWave, next_idx);
    next_idx = fetch_index(m0 + 2 * kWave);
    while (cur < nc) {
      const int s = cur_start > m0 ? cur_start - m0 : 0;
      const int e = cur_end < m0 + cnt ? cur_end - m0 : cnt;
      for (int t = s; t < e; t += 4 * kGatherAhead) {
        float g[kGatherAhead][kLive], w[kGatherAhead];
#pragma unroll
        for (int u = 0; u < kGatherAhead; ++u) {
          const int n = t + 4 * u + quarter;
          const int at = n < e ? n : s;   // past the point's pairs: its first one, weighted 0
          const char *row = grads + (size_t)stage->row[at] + 4 * col;
#pragma unroll
          for (int c = 0; c < kLive; ++c)
            g[u][c] = *reinterpret_cast<const float *>(
                row + (kWhole || 64u * c < last_channel ? 64u * c : last_channel));
          w[u] = n < e ? basis(stage->geo[at]) : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kGatherAhead; ++u)
#pragma unroll
          for (int c = 0; c < kLive; ++c) acc[c] = fmaf(w[u], g[u][c], acc[c]);
      }
      if (cur_end > m0 + cnt) break;      // goes on in the next chunk
      finish_point(cur);
      ++cur;
      cur_start = cur_end;
      cur_end = __builtin_amdgcn_readlane(my_end, cur < nc ? cur : nc - 1);
    }
  }
  for (; cur < nc; ++cur) finish_point(cur);      // trailing points without pairs
}

template <int kLive, int D, int kAct, bool kWhole>
__global__ void __launch_bounds__(256) mc_conv_gather_grads_kernel(
    int64_t n_pts, int run_len, const float *__restrict__ grads, unsigned row_bytes,
    const int2 *__restrict__ nbrs, const int *__restrict__ ranges, McParams<D> p,
    const int *__restrict__ out_rows, int live, int add, float *__restrict__ out) {
  __shared__ PairStage stages[kWavesPerBlock];
  const MlpBasis<D, kAct> basis(p);
  gather_grads_body<kLive, D, kWhole>(n_pts, run_len, reinterpret_cast<const char *>(grads),
                                      row_bytes, nbrs, ranges, p, basis, out_rows, live, add != 0,
                                      out, &stages[threadIdx.x / kWave]);
}

template <int kLive, int D, int kKind, bool kWhole>
__global__ void __launch_bounds__(256) kp_conv_gather_grads_kernel(
    int64_t n_pts, int run_len, const float *__restrict__ grads, unsigned row_bytes,
    const int2 *__restrict__ nbrs, const int *__restrict__ ranges, McParams<D> p,
    const float *__restrict__ kernel_points, int num_kp, float sigma,
    const int *__restrict__ out_rows, int live, float *__restrict__ out) {
  __shared__ PairStage stages[kWavesPerBlock];
  const KpBasis<D, kKind> basis(kernel_points, num_kp, sigma);
  gather_grads_body<kLive, D, kWhole>(n_pts, run_len, reinterpret_cast<const char *>(grads),
                                      row_bytes, nbrs, ranges, p, basis, out_rows, live, false,
                                      out, &stages[threadIdx.x / kWave]);
}

// As for the projection (mc_conv.hip): shorter runs on small inputs.
static int gather_run_len(int64_t n) {
  return n >= 160000 ? kGatherRun : n >= 64000 ? 4 : n >= 20000 ? 2 : 1;
}

static int check_gather_args(const char *op, int num_dims, int num_features, int padded_features,
                             int64_t num_centres, int64_t num_neighbors, int64_t num_pts) {
  MCCNN_REQUIRE(num_dims == 2 || num_dims == 3, "%s supports 2 and 3 dimensions (got %d)", op,
                num_dims);
  MCCNN_REQUIRE(num_features > 0 && num_features <= padded_features && num_features <= 16,
                "%s supports 1 to 16 channels (got %d of %d)", op, num_features, padded_features);
  MCCNN_REQUIRE(num_neighbors >= 0 && num_neighbors < ((int64_t)1 << 31) && num_pts >= 0 &&
                    num_pts < ((int64_t)1 << 31) && num_centres >= 0,
                "%s expects sizes in [0, 2^31)", op);
  MCCNN_REQUIRE(num_centres * padded_features * kFusedK < ((int64_t)1 << 30),
                "%s expects fewer than 2^30 values of the projection's gradient", op);
  return MCCNN_OK;
}

}  // namespace mccnn

using namespace mccnn;

extern "C" int mccnn_mc_conv_gather_grads(
    mccnn_stream_t stream, int num_dims, int64_t num_centres, const float *centres,
    int num_features, int padded_features, const float *projection_grads, int64_t num_pts,
    const float *points, int64_t num_neighbors, const int32_t *neighbors, const int32_t *ranges,
    const float *inv_radii, int num_mlps, int activation, const float *weights,
    const float *biases, const float *pdf, const int32_t *out_rows, int accumulate, float *out) {
  int rc = check_gather_args("mc_conv_gather_grads", num_dims, num_features, padded_features,
                             num_centres, num_neighbors, num_pts);
  if (rc != MCCNN_OK) return rc;
  MCCNN_REQUIRE(num_mlps > 0 && kFusedK % num_mlps == 0 && activation >= 0 && activation <= 2,
                "mc_conv_gather_grads expects kernel MLPs that divide 16 basis columns and a known "
                "activation");
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(ranges && out && points && inv_radii && weights && biases &&
                    (num_neighbors == 0 || (centres && projection_grads && neighbors && pdf)),
                "mc_conv_gather_grads received a null tensor");
  const int run_len = gather_run_len(num_pts);
  const dim3 grid(wave_grid((num_pts + run_len - 1) / run_len)), block(256);
#define MCCNN_GATHER(LIVE_, D_, WHOLE_)                                                         \
  {                                                                                             \
    McParams<D_> prm{centres, points, inv_radii, weights, biases, pdf, kFusedK / num_mlps,      \
                     activation};                                                               \
    MCCNN_ACT_SWITCH(activation,                                                                \
                     hipLaunchKernelGGL((mc_conv_gather_grads_kernel<LIVE_, D_, ACT, WHOLE_>),  \
                                        grid, block, 0, as_stream(stream), num_pts, run_len,    \
                                        projection_grads, 64u * padded_features,                \
                                        (const int2 *)neighbors, ranges, prm, out_rows,         \
                                        num_features, accumulate, out));                        \
  }
#define MCCNN_GATHER_D(LIVE_)                                                                   \
  if (padded_features >= LIVE_) {                                                               \
    if (num_dims == 3) MCCNN_GATHER(LIVE_, 3, true) else MCCNN_GATHER(LIVE_, 2, true)           \
  } else {                                                                                      \
    if (num_dims == 3) MCCNN_GATHER(LIVE_, 3, false) else MCCNN_GATHER(LIVE_, 2, false)         \
  }
  if (num_features <= 4) { MCCNN_GATHER_D(4) }
  else if (num_features <= 8) { MCCNN_GATHER_D(8) }
  else { MCCNN_GATHER_D(16) }
#undef MCCNN_GATHER_D
#undef MCCNN_GATHER
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_kp_conv_gather_grads(
    mccnn_stream_t stream, int num_dims, int64_t num_centres, const float *centres,
    int num_features, int padded_features, const float *projection_grads, int64_t num_pts,
    const float *points, int64_t num_neighbors, const int32_t *neighbors, const int32_t *ranges,
    const float *inv_radii, int num_kernel_points, const float *kernel_points, int kind,
    float sigma, const int32_t *out_rows, float *out) {
  int rc = check_gather_args("kp_conv_gather_grads", num_dims, num_features, padded_features,
                             num_centres, num_neighbors, num_pts);
  if (rc != MCCNN_OK) return rc;
  MCCNN_REQUIRE(num_kernel_points > 0 && num_kernel_points <= kFusedK,
                "kp_conv_gather_grads supports 1 to 16 kernel points (got %d)", num_kernel_points);
  MCCNN_REQUIRE((kind == 0 || kind == 1) && sigma > 0.0f,
                "kp_conv_gather_grads expects kind 0 (linear) or 1 (gaussian) and a positive sigma");
  if (num_pts == 0) return MCCNN_OK;
  MCCNN_REQUIRE(ranges && out && points && inv_radii && kernel_points &&
                    (num_neighbors == 0 || (centres && projection_grads && neighbors)),
                "kp_conv_gather_grads received a null tensor");
  const int run_len = gather_run_len(num_pts);
  const dim3 grid(wave_grid((num_pts + run_len - 1) / run_len)), block(256);
#define MCCNN_GATHER(LIVE_, D_, WHOLE_)                                                         \
  {                                                                                             \
    McParams<D_> prm{centres, points, inv_radii, nullptr, nullptr, nullptr, 1, 0};              \
    MCCNN_INFLUENCE_SWITCH(                                                                     \
        kind, sigma,                                                                            \
        hipLaunchKernelGGL((kp_conv_gather_grads_kernel<LIVE_, D_, KIND, WHOLE_>), grid, block, \
                           0, as_stream(stream), num_pts, run_len, projection_grads,            \
                           64u * padded_features, (const int2 *)neighbors, ranges, prm,         \
                           kernel_points, num_kernel_points, sigma, out_rows, num_features,     \
                           out));                                                               \
  }
#define MCCNN_GATHER_D(LIVE_)                                                                   \
  if (padded_features >= LIVE_) {                                                               \
    if (num_dims == 3) MCCNN_GATHER(LIVE_, 3, true) else MCCNN_GATHER(LIVE_, 2, true)           \
  } else {                                                                                      \
    if (num_dims == 3) MCCNN_GATHER(LIVE_, 3, false) else MCCNN_GATHER(LIVE_, 2, false)         \
  }
  if (num_features <= 4) { MCCNN_GATHER_D(4) }
  else if (num_features <= 8) { MCCNN_GATHER_D(8) }
  else { MCCNN_GATHER_D(16) }
#undef MCCNN_GATHER_D
#undef MCCNN_GATHER
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}
