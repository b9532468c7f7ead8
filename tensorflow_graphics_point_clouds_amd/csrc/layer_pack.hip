// Operand preparation of the convolution layers: channel padding, and the forms of a
// layer's weights that its kernels read.
//
// The layer kernels work on 16 / 32 / 64 / 128 channels, multiples of 16 output columns and
// 16 / 32 / 64 basis columns, and on the final weights as one dense matrix in up to four
// orders (forward and feature-gradient product, each natural or transposed).  Composed from
// tensor operations that is a pad, a block scatter, two permutations and their copies per
// pass -- ten launches of 4 to 5 us each around kernels that take as long on a small cloud;
// here it is one launch per direction.  All of it is a few hundred kilobytes: bound by the
// launch.
#include "common.h"
#include "fill.h"

namespace mccnn {

// out[i, c] = src[rows[i], col0 + c] for c < cols, 0 for cols <= c < out_cols.  `kVec`: four
// columns per thread (cols, ld, col0 and out_cols multiples of 4).
template <bool kVec>
__global__ void __launch_bounds__(256) gather_rows_padded_kernel(
    int64_t total, int out_units, int unit_cols, int64_t ld, const float *__restrict__ src,
    const int *__restrict__ rows, float *__restrict__ out) {
  for (int64_t t = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; t < total;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = t / out_units;
    const int u = (int)(t - i * out_units);
    const int64_t row = rows ? rows[i] : i;
    if (kVec) {
      float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if (u < unit_cols) v = reinterpret_cast<const float4 *>(src + row * ld)[u];
      reinterpret_cast<float4 *>(out)[t] = v;
    } else {
      out[t] = u < unit_cols ? src[row * ld + u] : 0.0f;
    }
  }
}

struct LayerShapeArgs {
  int C, H, G;            // of the caller's weights [L, C*H, G]
  int first, mlps;        // the kernel MLPs first .. first + mlps - 1 form this layer
  int Cp, Hp, Gp;         // padded
};

// Element (c, k = m Hp + h, f = m' Gp + g) of the dense matrix: zero off the diagonal blocks.
__device__ __forceinline__ float dense_element(const LayerShapeArgs &a,
                                               const float *__restrict__ w, int c, int k, int f) {
  const int m = k / a.Hp, h = k - m * a.Hp, mf = f / a.Gp, g = f - mf * a.Gp;
  if (m != mf || c >= a.C || h >= a.H || g >= a.G) return 0.0f;
  return w[((int64_t)(a.first + m) * a.C * a.H + (int64_t)c * a.H + h) * a.G + g];
}

// w [(c,k), f], wt [f, (c,k)], w2 [(f,k), c], w2t [c, (f,k)] (each may be null), and the
// kernel MLPs' weights kw [mlps, D, Hp], kb [mlps * Hp].
__global__ void __launch_bounds__(256) pack_layer_weights_kernel(
    LayerShapeArgs a, int D, const float *__restrict__ src, const float *__restrict__ kw_src,
    const float *__restrict__ kb_src, float *__restrict__ w, float *__restrict__ wt,
    float *__restrict__ w2, float *__restrict__ w2t, float *__restrict__ kw,
    float *__restrict__ kb, float *__restrict__ all) {
  const int K = a.mlps * a.Hp, F = a.mlps * a.Gp, size = a.Cp * K * F;
  const int which = blockIdx.y, part = blockIdx.z;      // (a part: the next `mlps` kernel MLPs)
  if (which == 5) {                                     // all of them as one dense matrix [(c,k), f]
    const int parts = gridDim.z, Fa = parts * F, Ka = parts * K;
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < size * parts;
         t += gridDim.x * blockDim.x) {
      const int e = part * size * parts + t;            // a part's share of the size * parts^2
      all[e] = dense_element(a, src, e / Fa / Ka, e / Fa % Ka, e % Fa);
    }
    return;
  }
  a.first += part * a.mlps;
  float *dst = which == 0 ? w : which == 1 ? wt : which == 2 ? w2 : which == 3 ? w2t : nullptr;
  if (dst) dst += (int64_t)part * size;
  if (kw) {
    kw += part * D * K;
    kb += part * K;
  }
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < size; t += gridDim.x * blockDim.x) {
    if (dst == nullptr) break;
    int c, k, f;
    if (which == 0) {
      f = t % F; k = t / F % K; c = t / F / K;
    } else if (which == 1) {
      k = t % K; c = t / K % a.Cp; f = t / K / a.Cp;
    } else if (which == 2) {
      c = t % a.Cp; k = t / a.Cp % K; f = t / a.Cp / K;
    } else {
      k = t % K; f = t / K % F; c = t / K / F;
    }
    dst[t] = dense_element(a, src, c, k, f);
  }
  if (which == 4 && blockIdx.x == 0) {
    for (int t = threadIdx.x; t < D * K; t += blockDim.x) {      // kw[m][d][h]
      const int h = t % a.Hp, d = t / a.Hp % D, m = t / a.Hp / D;
      kw[t] = h < a.H ? kw_src[((a.first + m) * D + d) * a.H + h] : 0.0f;
    }
    for (int t = threadIdx.x; t < K; t += blockDim.x) {
      const int h = t % a.Hp, m = t / a.Hp;
      kb[t] = h < a.H ? kb_src[(a.first + m) * a.H + h] : 0.0f;
    }
  }
}

// The gradients back in the caller's shapes: final-weight gradient from the product's
// [Cp, (f, k)] or [f, (c, k)] result (element (c, f, k) at c c_stride + f f_stride + k), kernel-MLP
// gradients from [mlps, D, Hp] and [mlps * Hp].
__global__ void __launch_bounds__(256) unpack_layer_grads_kernel(
    LayerShapeArgs a, int D, int c_stride, int f_stride, const float *__restrict__ ddense,
    const float *__restrict__ dkw_src, const float *__restrict__ dkb_src,
    float *__restrict__ dfinal, float *__restrict__ dkw, float *__restrict__ dkb) {
  const int per = a.C * a.H * a.G, size = a.mlps * per, part = blockIdx.z;
  a.first += part * a.mlps;                    // (f of the parts one after the other)
  ddense += (int64_t)part * a.mlps * a.Gp * f_stride;
  dkw_src += part * D * a.mlps * a.Hp;
  dkb_src += part * a.mlps * a.Hp;
  if (dfinal)
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < size; t += gridDim.x * blockDim.x) {
      const int g = t % a.G, h = t / a.G % a.H, c = t / a.G / a.H % a.C, m = t / per;
      dfinal[(int64_t)a.first * per + t] =
          ddense[(int64_t)c * c_stride + (int64_t)(m * a.Gp + g) * f_stride + m * a.Hp + h];
    }
  if (blockIdx.x == 0 && dkw) {
    for (int t = threadIdx.x; t < a.mlps * D * a.H; t += blockDim.x) {
      const int h = t % a.H, d = t / a.H % D, m = t / a.H / D;
      dkw[a.first * D * a.H + t] = dkw_src[(m * D + d) * a.Hp + h];
    }
    for (int t = threadIdx.x; t < a.mlps * a.H; t += blockDim.x)
      dkb[a.first * a.H + t] = dkb_src[t / a.H * a.Hp + t % a.H];
  }
}

static int check_shape(const char *op, const LayerShapeArgs &a) {
  MCCNN_REQUIRE(a.C > 0 && a.H > 0 && a.G > 0 && a.first >= 0 && a.mlps > 0 && a.Cp >= a.C &&
                    a.Hp >= a.H && a.Gp >= a.G,
                "%s expects padded sizes of at least the given ones", op);
  MCCNN_REQUIRE((int64_t)a.Cp * a.mlps * a.Hp * a.mlps * a.Gp < ((int64_t)1 << 28),
                "%s expects fewer than 2^28 weights", op);
  return MCCNN_OK;
}

}  // namespace mccnn

using namespace mccnn;

extern "C" int mccnn_gather_rows_padded(mccnn_stream_t stream, int64_t num_rows,
                                        const int32_t *rows, const float *src, int64_t src_stride,
                                        int first_col, int num_cols, int num_cols_out,
                                        float *out) {
  MCCNN_REQUIRE(num_rows >= 0, "gather_rows_padded expects a non-negative size");
  MCCNN_REQUIRE(num_cols > 0 && num_cols_out >= num_cols && first_col >= 0 &&
                    src_stride >= (int64_t)first_col + num_cols,
                "gather_rows_padded expects 0 < num_cols <= num_cols_out and columns inside a row");
  if (num_rows == 0) return MCCNN_OK;
  MCCNN_REQUIRE(src && out, "gather_rows_padded received a null tensor");
  const bool vec = num_cols % 4 == 0 && num_cols_out % 4 == 0 && src_stride % 4 == 0 &&
                   first_col % 4 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(out) % 16 == 0;
  const int unit = vec ? 4 : 1;
  const int64_t total = num_rows * (num_cols_out / unit);
  const unsigned grid = blocks_for(total > ((int64_t)1 << 26) ? (int64_t)1 << 26 : total, 256);
  if (vec)
    hipLaunchKernelGGL(gather_rows_padded_kernel<true>, dim3(grid), dim3(256), 0,
                       as_stream(stream), total, num_cols_out / 4, num_cols / 4, src_stride,
                       src + first_col, rows, out);
  else
    hipLaunchKernelGGL(gather_rows_padded_kernel<false>, dim3(grid), dim3(256), 0,
                       as_stream(stream), total, num_cols_out, num_cols, src_stride,
                       src + first_col, rows, out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

static int pack_layer_weights(mccnn_stream_t stream, int num_dims, const LayerShapeArgs &a,
                              int parts, const float *final_weights, const float *kernel_weights,
                              const float *kernel_biases, float *w_out, float *wt_out,
                              float *w2_out, float *w2t_out, float *kernel_weights_out,
                              float *kernel_biases_out, float *all_out) {
  int rc = check_shape("pack_layer_weights", a);
  if (rc != MCCNN_OK) return rc;
  const bool kernel = kernel_weights_out != nullptr;
  MCCNN_REQUIRE(final_weights && (!kernel || (kernel_weights && kernel_biases &&
                                              kernel_biases_out)),
                "pack_layer_weights received a null tensor");
  const int64_t size = (int64_t)a.Cp * a.mlps * a.Hp * a.mlps * a.Gp;
  MCCNN_REQUIRE(size * parts * parts < ((int64_t)1 << 28),
                "pack_layer_weights expects fewer than 2^28 weights");
  const unsigned grid = blocks_for(size > (1 << 20) ? (1 << 20) : size, 256);
  const unsigned outputs = all_out ? 6 : kernel ? 5 : w2t_out ? 4 : w2_out ? 3 : wt_out ? 2 : 1;
  hipLaunchKernelGGL(pack_layer_weights_kernel, dim3(grid, outputs, (unsigned)parts), dim3(256), 0,
                     as_stream(stream), a, num_dims, final_weights, kernel_weights, kernel_biases,
                     w_out, wt_out, w2_out, w2t_out, kernel_weights_out, kernel_biases_out,
                     all_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_pack_layer_weights(mccnn_stream_t stream, int num_dims, int num_features,
                                        int hidden, int group_features, int first_mlp,
                                        int num_mlps, int padded_features, int padded_hidden,
                                        int padded_group, const float *final_weights,
                                        const float *kernel_weights, const float *kernel_biases,
                                        float *w_out, float *wt_out, float *w2_out,
                                        float *w2t_out, float *kernel_weights_out,
                                        float *kernel_biases_out) {
  const LayerShapeArgs a = {num_features, hidden, group_features, first_mlp, num_mlps,
                            padded_features, padded_hidden, padded_group};
  return pack_layer_weights(stream, num_dims, a, 1, final_weights, kernel_weights, kernel_biases,
                            w_out, wt_out, w2_out, w2t_out, kernel_weights_out, kernel_biases_out,
                            nullptr);
}

extern "C" int mccnn_pack_layer_weights_pair(
    mccnn_stream_t stream, int num_dims, int num_features, int hidden, int group_features,
    int num_mlps, int padded_features, int padded_hidden, int padded_group,
    const float *final_weights, const float *kernel_weights, const float *kernel_biases,
    float *w_out, float *w2_out, float *kernel_weights_out, float *kernel_biases_out,
    float *all_out) {
  const LayerShapeArgs a = {num_features, hidden, group_features, 0, num_mlps,
                            padded_features, padded_hidden, padded_group};
  return pack_layer_weights(stream, num_dims, a, 2, final_weights, kernel_weights, kernel_biases,
                            w_out, nullptr, w2_out, nullptr, kernel_weights_out, kernel_biases_out,
                            all_out);
}

static int unpack_layer_grads(mccnn_stream_t stream, int num_dims, const LayerShapeArgs &a,
                              bool by_output, const float *dense_grads,
                              const float *kernel_weight_grads, const float *kernel_bias_grads,
                              float *final_grads_out, float *weight_grads_out,
                              float *bias_grads_out, int parts = 1) {
  int rc = check_shape("unpack_layer_grads", a);
  if (rc != MCCNN_OK) return rc;
  MCCNN_REQUIRE((!final_grads_out || dense_grads) &&
                    (!weight_grads_out || (kernel_weight_grads && kernel_bias_grads &&
                                           bias_grads_out)),
                "unpack_layer_grads received a null tensor");
  const int64_t size = (int64_t)a.mlps * a.C * a.H * a.G;
  const unsigned grid = blocks_for(size > (1 << 20) ? (1 << 20) : size, 256);
  const int K = a.mlps * a.Hp, F = a.mlps * a.Gp;
  hipLaunchKernelGGL(unpack_layer_grads_kernel, dim3(grid, 1, (unsigned)parts), dim3(256), 0,
                     as_stream(stream), a, num_dims, by_output ? K : parts * F * K,
                     by_output ? a.Cp * K : K, dense_grads, kernel_weight_grads,
                     kernel_bias_grads, final_grads_out, weight_grads_out, bias_grads_out);
  MCCNN_LAUNCH_CHECK();
  return MCCNN_OK;
}

extern "C" int mccnn_unpack_layer_grads(mccnn_stream_t stream, int num_dims, int num_features,
                                        int hidden, int group_features, int first_mlp,
                                        int num_mlps, int padded_features, int padded_hidden,
                                        int padded_group, const float *dense_grads,
                                        const float *kernel_weight_grads,
                                        const float *kernel_bias_grads, float *final_grads_out,
                                        float *weight_grads_out, float *bias_grads_out) {
  const LayerShapeArgs a = {num_features, hidden, group_features, first_mlp, num_mlps,
                            padded_features, padded_hidden, padded_group};
  return unpack_layer_grads(stream, num_dims, a, false, dense_grads, kernel_weight_grads,
                            kernel_bias_grads, final_grads_out, weight_grads_out, bias_grads_out);
}

extern "C" int mccnn_unpack_layer_grads_wt(mccnn_stream_t stream, int num_dims, int num_features,
                                           int hidden, int group_features, int first_mlp,
                                           int num_mlps, int padded_features, int padded_hidden,
                                           int padded_group, const float *dense_grads,
                                           const float *kernel_weight_grads,
                                           const float *kernel_bias_grads, float *final_grads_out,
                                           float *weight_grads_out, float *bias_grads_out) {
  const LayerShapeArgs a = {num_features, hidden, group_features, first_mlp, num_mlps,
                            padded_features, padded_hidden, padded_group};
  return unpack_layer_grads(stream, num_dims, a, true, dense_grads, kernel_weight_grads,
                            kernel_bias_grads, final_grads_out, weight_grads_out, bias_grads_out);
}

extern "C" int mccnn_unpack_layer_grads_pair(
    mccnn_stream_t stream, int num_dims, int num_features, int hidden, int group_features,
    int num_mlps, int padded_features, int padded_hidden, int padded_group,
    const float *dense_grads, const float *kernel_weight_grads, const float *kernel_bias_grads,
    float *final_grads_out, float *weight_grads_out, float *bias_grads_out) {
  const LayerShapeArgs a = {num_features, hidden, group_features, 0, num_mlps,
                            padded_features, padded_hidden, padded_group};
  return unpack_layer_grads(stream, num_dims, a, false, dense_grads, kernel_weight_grads,
                            kernel_bias_grads, final_grads_out, weight_grads_out, bias_grads_out, 2);
}
