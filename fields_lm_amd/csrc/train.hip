// train.hip — the Field block's elementwise work in training, forward and backward (reference:
// src/fields_official/reference/field_only_v4_chunked_triton_wiki100.py, "canon"): the RMSNorms
// (300-309), the gated residual with the norm after it (1193-1195, 1219-1221), SwiGLU (312-325) and
// the transition parameters (1169-1173). The residual stream, read and all maths are fp32; what goes to
// or comes from a product is of that product's type.
//
// All of them are bound by memory: each tensor is read and written once, 16 bytes per lane and access
// (8 for fp32 twice), one wave per row, where the stock ops made six to ten passes each way. Weight
// gradients: a wave adds its rows in registers, a block its waves in LDS, and a second launch the blocks,
// in a fixed order. 4,096 tokens, dim 1,024, bf16 autocast: read_norm 12.0 us forward and 22.3 + 4.3 us
// backward (fp32 [4096, 2048]: 50 MB and 84 MB), gated residual and norm 11.0 and 18.4 + 4.3 us, SwiGLU
// backward 17.3 us; a training pass of the block 865 us of kernels in 57 launches (stock ops: 1,416 in 144).
#include "fl_common.h"

namespace {

using namespace fl;

constexpr int kGradBlocks = 256;  // blocks of a backward launch (4 waves each), and partial rows it leaves

template <typename T>
__device__ __forceinline__ float sigmoid(float x);
template <>
__device__ __forceinline__ float sigmoid<float>(float x) { return 1.0f / (1.0f + expf(-x)); }
template <>
__device__ __forceinline__ float sigmoid<bf16_bits>(float x) { return sigmoid_bf16(x); }

// out = (x rsqrt(mean x^2 + eps)) w; GATED: x_new = x + round(out_in * round(sigmoid(g))) first (in the
// products' type G) and its norm. rstd is kept for the backward.
template <typename G, typename OT, bool GATED, int NV>
__global__ __launch_bounds__(256) void fl_train_norm_kernel(
    const float* __restrict__ x, const G* __restrict__ prod, const G* __restrict__ gate, int64_t rows, int dim,
    const float* __restrict__ w, float eps, float inv_dim, float* __restrict__ x_new, OT* __restrict__ out,
    float* __restrict__ rstd) {
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int64_t base = row * dim;
  float v[NV][8], acc = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c < dim) {
      Vec<float, 8>::load(x + base + c, v[i]);
      if constexpr (GATED) {
        float o[8], g[8];
        Vec<G, 8>::load(prod + base + c, o);
        Vec<G, 8>::load(gate + base + c, g);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] += round_as<G>(o[j] * round_as<G>(sigmoid<G>(g[j])));
        Vec<float, 8>::store(x_new + base + c, v[i]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fmaf(v[i][j], v[i][j], acc);
    }
  }
  const float scale = rsqrtf(fmaf(wave_sum(acc), inv_dim, eps));
  if (lane == 0) rstd[row] = scale;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c < dim) {
      float ww[8];
      Vec<float, 8>::load(w + c, ww);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = (v[i][j] * scale) * ww[j];
      Vec<OT, 8>::store(out + base + c, v[i]);
    }
  }
}

// With xh = x rstd and t = gy w: gx = rstd (t - xh mean(t xh)), gw = sum over rows of gy xh.
// GATED: x is x_new, gx adds the residual's own gradient, and with s = sigmoid(g):
// g_prod = gx s, g_gate = gx prod s (1 - s).
template <typename G, typename OT, bool GATED, int NV>
__global__ __launch_bounds__(256) void fl_train_norm_backward_kernel(
    const OT* __restrict__ gy, const float* __restrict__ gres, const float* __restrict__ x,
    const G* __restrict__ prod, const G* __restrict__ gate, int64_t rows, int dim, const float* __restrict__ w,
    const float* __restrict__ rstd, float inv_dim, float* __restrict__ gx, G* __restrict__ g_prod,
    G* __restrict__ g_gate, float* __restrict__ part) {
  extern __shared__ float s_part[];  // [4][dim]
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6);
  float ww[NV][8], gw[NV][8];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * 64 + lane) * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) ww[i][j] = gw[i][j] = 0.f;
    if (c < dim) Vec<float, 8>::load(w + c, ww[i]);
  }
  for (int64_t row = (int64_t)blockIdx.x * 4 + wave; row < rows; row += (int64_t)gridDim.x * 4) {
    const int64_t base = row * dim;
    const float rs = rstd[row];
    float xh[NV][8], t[NV][8], acc = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = (i * 64 + lane) * 8;
      if (c < dim) {
        float g[8];
        Vec<float, 8>::load(x + base + c, xh[i]);
        Vec<OT, 8>::load(gy + base + c, g);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          xh[i][j] *= rs;
          gw[i][j] = fmaf(g[j], xh[i][j], gw[i][j]);
          t[i][j] = g[j] * ww[i][j];
          acc = fmaf(t[i][j], xh[i][j], acc);
        }
      }
    }
    const float mean = wave_sum(acc) * inv_dim;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = (i * 64 + lane) * 8;
      if (c < dim) {
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = rs * fmaf(-xh[i][j], mean, t[i][j]);
        if constexpr (GATED) {
          float r[8], p[8], g[8], gp[8], gg[8];
          Vec<float, 8>::load(gres + base + c, r);
          Vec<G, 8>::load(prod + base + c, p);
          Vec<G, 8>::load(gate + base + c, g);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            o[j] += r[j];
            const float s = sigmoid<G>(g[j]);
            gp[j] = o[j] * s;
            gg[j] = o[j] * p[j] * s * (1.0f - s);
          }
          Vec<G, 8>::store(g_prod + base + c, gp);
          Vec<G, 8>::store(g_gate + base + c, gg);
        }
        Vec<float, 8>::store(gx + base + c, o);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c < dim) Vec<float, 8>::store(s_part + wave * dim + c, gw[i]);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < dim; c += 256)
    part[(int64_t)blockIdx.x * dim + c] = ((s_part[c] + s_part[dim + c]) + s_part[2 * dim + c]) + s_part[3 * dim + c];
}

// column sums of part [n, dim]: 64 columns per block, 16 waves each a run of rows
__global__ __launch_bounds__(1024) void fl_column_sum_kernel(const float* __restrict__ part, int n, int dim,
                                                             float* __restrict__ out) {
  __shared__ float s_sum[16][64];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), c = blockIdx.x * 64 + lane;
  const int per = (n + 15) / 16, r0 = min(wave * per, n), r1 = min(r0 + per, n);
  float acc = 0.f;
  if (c < dim) {
#pragma unroll 8
    for (int r = r0; r < r1; ++r) acc += part[(int64_t)r * dim + c];
  }
  s_sum[wave][lane] = acc;
  __syncthreads();
  if (wave == 0 && c < dim) {
    float t = 0.f;
#pragma unroll
    for (int u = 0; u < 16; ++u) t += s_sum[u][lane];
    out[c] = t;
  }
}

// [gate | up] and dL/d(silu(gate) up) -> [dgate | dup]
template <typename T>
__global__ __launch_bounds__(256) void fl_swiglu_backward_kernel(const T* __restrict__ gu, const T* __restrict__ gy,
                                                                 uint32_t n_vec, uint32_t row_vecs, int hidden,
                                                                 T* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n_vec) return;
  const uint32_t r = i / row_vecs;
  const int64_t at = (int64_t)r * hidden + (int64_t)i * 8;
  float g[8], u[8], d[8], dg[8], du[8];
  Vec<T, 8>::load(gu + at, g);
  Vec<T, 8>::load(gu + at + hidden, u);
  Vec<T, 8>::load(gy + (int64_t)i * 8, d);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float s = sigmoid<T>(g[j]), a = g[j] * s;
    du[j] = d[j] * a;
    dg[j] = d[j] * u[j] * fmaf(a, 1.0f - s, s);  // silu' = s + g s (1 - s)
  }
  Vec<T, 8>::store(out + at, dg);
  Vec<T, 8>::store(out + at + hidden, du);
}

// Gradients through radius = clamp(sigmoid(l), 0.5, 0.99995), tr = radius cos(theta), ti = radius
// sin(theta), gamma = sqrt(max(1 - radius^2, 1e-4)); both clamps pass the gradient at their bounds.
__global__ __launch_bounds__(256) void fl_field_params_backward_kernel(
    const float* __restrict__ radius_logit, const float* __restrict__ theta, int C, const float* __restrict__ gtr,
    const float* __restrict__ gti, const float* __restrict__ ggamma, float* __restrict__ g_logit,
    float* __restrict__ g_theta) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= C) return;
  const float s = 1.0f / (1.0f + expf(-radius_logit[i])), r = s != s ? s : fminf(fmaxf(s, 0.50f), 0.99995f);
  const float c = cosf(theta[i]), n = sinf(theta[i]), d = 1.0f - r * r;
  float gr = fmaf(gtr[i], c, gti[i] * n);
  if (!(d < 1e-4f)) gr -= ggamma[i] * r / sqrtf(d);
  g_logit[i] = s < 0.50f || s > 0.99995f ? 0.f : gr * s * (1.0f - s);
  g_theta[i] = r * fmaf(gti[i], c, -(gtr[i] * n));
}

bool norm_args_ok(int64_t rows, int64_t dim) {
  return rows > 0 && rows <= ((int64_t)1 << 31) - 1 && dim > 0 && dim % 8 == 0 && dim <= 4096;
}

bool vec_ok(const void* p) { return p != nullptr && aligned(p, 16); }

size_t part_bytes(int64_t dim) { return (size_t)kGradBlocks * dim * 4; }

template <typename G, typename OT, bool GATED>
int norm_forward(const float* x, const void* prod, const void* gate, int64_t rows, int64_t dim, const float* w,
                 float eps, float* x_new, void* out, float* rstd, hipStream_t s) {
  const float inv = (float)(1.0 / (double)dim);
#define FL_TN(NV)                                                                                             \
  fl_train_norm_kernel<G, OT, GATED, NV><<<(unsigned)cdiv(rows, 4), 256, 0, s>>>(                             \
      x, static_cast<const G*>(prod), static_cast<const G*>(gate), rows, (int)dim, w, eps, inv, x_new,        \
      static_cast<OT*>(out), rstd)
  if (dim <= 1024) FL_TN(2);
  else if (dim <= 2048) FL_TN(4);
  else FL_TN(8);
#undef FL_TN
  return hip_status(hipGetLastError());
}

template <typename G, typename OT, bool GATED>
int norm_backward(const void* gy, const float* gres, const float* x, const void* prod, const void* gate, int64_t rows,
                  int64_t dim, const float* w, const float* rstd, float* gx, void* g_prod, void* g_gate, float* gw,
                  float* part, hipStream_t s) {
  const float inv = (float)(1.0 / (double)dim);
  const int64_t want = cdiv(rows, 4);
  const int blocks = (int)(want < kGradBlocks ? want : kGradBlocks);
#define FL_TB(NV)                                                                                             \
  fl_train_norm_backward_kernel<G, OT, GATED, NV><<<(unsigned)blocks, 256, (unsigned)(4 * dim * 4), s>>>(     \
      static_cast<const OT*>(gy), gres, x, static_cast<const G*>(prod), static_cast<const G*>(gate), rows,    \
      (int)dim, w, rstd, inv, gx, static_cast<G*>(g_prod), static_cast<G*>(g_gate), part)
  if (dim <= 1024) FL_TB(2);
  else if (dim <= 2048) FL_TB(4);
  else FL_TB(8);
#undef FL_TB
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_status(e);
  fl_column_sum_kernel<<<(unsigned)cdiv(dim, 64), 1024, 0, s>>>(part, blocks, (int)dim, gw);
  return hip_status(hipGetLastError());
}

}  // namespace

extern "C" {

size_t fl_train_workspace_bytes(int64_t dim) { return dim > 0 ? part_bytes(dim) : 0; }

int fl_train_norm(const float* x, int64_t rows, int64_t dim, const float* weight, float eps, void* out, int out_dtype,
                  float* rstd, void* stream) {
  if (!dtype_ok(out_dtype)) return FL_ERR_DTYPE;
  if (!norm_args_ok(rows, dim) || !vec_ok(x) || !vec_ok(weight) || !vec_ok(out) || !rstd || !aligned(rstd, 4) ||
      !(eps >= 0.f))
    return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return out_dtype == FL_DTYPE_BF16
             ? norm_forward<float, bf16_bits, false>(x, nullptr, nullptr, rows, dim, weight, eps, nullptr, out, rstd, s)
             : norm_forward<float, float, false>(x, nullptr, nullptr, rows, dim, weight, eps, nullptr, out, rstd, s);
}

int fl_train_norm_backward(const void* gy, int gy_dtype, const float* x, int64_t rows, int64_t dim,
                           const float* weight, const float* rstd, float* gx, float* gw, void* workspace,
                           size_t workspace_bytes, void* stream) {
  if (!dtype_ok(gy_dtype)) return FL_ERR_DTYPE;
  if (!norm_args_ok(rows, dim) || !vec_ok(gy) || !vec_ok(x) || !vec_ok(weight) || !rstd || !aligned(rstd, 4) ||
      !vec_ok(gx) || !gw || !aligned(gw, 4))
    return FL_ERR_INVALID_ARGUMENT;
  if (!workspace || workspace_bytes < part_bytes(dim)) return FL_ERR_WORKSPACE;
  if (!aligned(workspace, 4)) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* part = static_cast<float*>(workspace);
  return gy_dtype == FL_DTYPE_BF16
             ? norm_backward<float, bf16_bits, false>(gy, nullptr, x, nullptr, nullptr, rows, dim, weight, rstd, gx,
                                                      nullptr, nullptr, gw, part, s)
             : norm_backward<float, float, false>(gy, nullptr, x, nullptr, nullptr, rows, dim, weight, rstd, gx,
                                                  nullptr, nullptr, gw, part, s);
}

int fl_train_gate_norm(const float* x, const void* out, const void* gate, int g_dtype, int64_t rows, int64_t dim,
                       const float* weight, float eps, float* x_new, void* normed, int normed_dtype, float* rstd,
                       void* stream) {
  if (!dtype_ok(g_dtype) || !dtype_ok(normed_dtype)) return FL_ERR_DTYPE;
  if (!norm_args_ok(rows, dim) || !vec_ok(x) || !vec_ok(out) || !vec_ok(gate) || !vec_ok(weight) || !vec_ok(x_new) ||
      !vec_ok(normed) || !rstd || !aligned(rstd, 4) || !(eps >= 0.f))
    return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define FL_GN(G, O) return norm_forward<G, O, true>(x, out, gate, rows, dim, weight, eps, x_new, normed, rstd, s);
  const bool g16 = g_dtype == FL_DTYPE_BF16, o16 = normed_dtype == FL_DTYPE_BF16;
  if (g16 && o16) FL_GN(bf16_bits, bf16_bits)
  if (g16) FL_GN(bf16_bits, float)
  if (o16) FL_GN(float, bf16_bits)
  FL_GN(float, float)
#undef FL_GN
}

int fl_train_gate_norm_backward(const float* g_x_new, const void* g_normed, int normed_dtype, const float* x_new,
                                const void* out, const void* gate, int g_dtype, int64_t rows, int64_t dim,
                                const float* weight, const float* rstd, float* gx, void* g_out, void* g_gate,
                                float* gw, void* workspace, size_t workspace_bytes, void* stream) {
  if (!dtype_ok(g_dtype) || !dtype_ok(normed_dtype)) return FL_ERR_DTYPE;
  if (!norm_args_ok(rows, dim) || !vec_ok(g_x_new) || !vec_ok(g_normed) || !vec_ok(x_new) || !vec_ok(out) ||
      !vec_ok(gate) || !vec_ok(weight) || !rstd || !aligned(rstd, 4) || !vec_ok(gx) || !vec_ok(g_out) ||
      !vec_ok(g_gate) || !gw || !aligned(gw, 4))
    return FL_ERR_INVALID_ARGUMENT;
  if (!workspace || workspace_bytes < part_bytes(dim)) return FL_ERR_WORKSPACE;
  if (!aligned(workspace, 4)) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* part = static_cast<float*>(workspace);
#define FL_GB(G, O)                                                                                          \
  return norm_backward<G, O, true>(g_normed, g_x_new, x_new, out, gate, rows, dim, weight, rstd, gx, g_out,  \
                                   g_gate, gw, part, s);
  const bool g16 = g_dtype == FL_DTYPE_BF16, o16 = normed_dtype == FL_DTYPE_BF16;
  if (g16 && o16) FL_GB(bf16_bits, bf16_bits)
  if (g16) FL_GB(bf16_bits, float)
  if (o16) FL_GB(float, bf16_bits)
  FL_GB(float, float)
#undef FL_GB
}

int fl_swiglu_backward(const void* gate_up, const void* gy, int dtype, int64_t rows, int64_t hidden, void* g_gate_up,
                       void* stream) {
  if (!dtype_ok(dtype)) return FL_ERR_DTYPE;
  if (rows <= 0 || hidden <= 0 || hidden % 8 || hidden > ((int64_t)1 << 30) ||
      rows * hidden / 8 >= ((int64_t)1 << 31))
    return FL_ERR_INVALID_ARGUMENT;
  if (!vec_ok(gate_up) || !vec_ok(gy) || !vec_ok(g_gate_up)) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int64_t n = rows * hidden / 8;
#define FL_SB(T)                                                                                             \
  fl_swiglu_backward_kernel<T><<<(unsigned)cdiv(n, 256), 256, 0, s>>>(                                       \
      static_cast<const T*>(gate_up), static_cast<const T*>(gy), (uint32_t)n, (uint32_t)(hidden / 8),        \
      (int)hidden, static_cast<T*>(g_gate_up))
  if (dtype == FL_DTYPE_BF16) FL_SB(bf16_bits);
  else FL_SB(float);
#undef FL_SB
  return hip_status(hipGetLastError());
}

int fl_field_params_backward(const float* radius_logit, const float* theta, int64_t C, const float* gtr,
                             const float* gti, const float* ggamma, float* g_logit, float* g_theta, void* stream) {
  if (C <= 0 || C > ((int64_t)1 << 24)) return FL_ERR_INVALID_ARGUMENT;
  if (!radius_logit || !theta || !gtr || !gti || !ggamma || !g_logit || !g_theta) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(radius_logit, 4) || !aligned(theta, 4) || !aligned(gtr, 4) || !aligned(gti, 4) ||
      !aligned(ggamma, 4) || !aligned(g_logit, 4) || !aligned(g_theta, 4))
    return FL_ERR_INVALID_ARGUMENT;
  fl_field_params_backward_kernel<<<(unsigned)cdiv(C, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      radius_logit, theta, (int)C, gtr, gti, ggamma, g_logit, g_theta);
  return hip_status(hipGetLastError());
}

}  // extern "C"
