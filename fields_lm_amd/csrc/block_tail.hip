// block_tail.hip — the Field block's elementwise work around its GEMMs and its scan
// (reference: src/fields_official/reference/field_only_v4_chunked_triton_wiki100.py, "canon"):
//   fl_gate_residual_norm   canon:1193-1195 and 1219-1221, RMSNorm 300-309
//   fl_swiglu               canon:312-325
// Each value is rounded exactly where the stock ops round it: an op on bf16 tensors computes in
// fp32 and rounds its result to bf16.
#include "fl_common.h"

namespace {

using namespace fl;

// sigmoid and silu of a loaded T: of a bf16 value the forms of fl_common.h, whose bf16 roundings are the
// library forms' for every input (a plain quotient of silu would miss 5.9375, so it takes the residual
// step); fp32 keeps the library exponential and division.
template <typename T>
__device__ __forceinline__ float sigmoid(float x);
template <>
__device__ __forceinline__ float sigmoid<float>(float x) { return 1.0f / (1.0f + expf(-x)); }
template <>
__device__ __forceinline__ float sigmoid<bf16_bits>(float x) { return sigmoid_bf16(x); }
template <typename T>
__device__ __forceinline__ float silu(float x);
template <>
__device__ __forceinline__ float silu<float>(float x) { return x / (1.0f + expf(-x)); }
template <>
__device__ __forceinline__ float silu<bf16_bits>(float x) { return silu_precise(x); }

// N norm weights of either type as fp32
template <int N>
__device__ __forceinline__ void load_weight(const void* w, int w16, int c, float* o) {
  if (w16) {
    Vec<bf16_bits, N>::load(static_cast<const bf16_bits*>(w) + c, o);
  } else {
    Vec<float, N>::load(static_cast<const float*>(w) + c, o);
  }
}

// ------------------------------------------------------------------------------------------
// gate = sigmoid(g), prod = out * gate (in the GEMM output type G), x1 = x + prod (in the
// residual type X), h = RMSNorm(x1) * w (fp32 math, rounded to X).
// Bound by memory at prefill sizes (five [rows, dim] streams) and by the launch at decode sizes.
// One wave per row, 16 bytes per lane and access with N = 8 (bf16), four rows per block. The sum of squares keeps one
// order for every N and launch shape: 256 strided chains over the row (c = i, i + 256, ...), each
// 64 of them added by a butterfly, the four sums in sequence; the row's values reach their chains
// through LDS (RES floats per wave; longer rows in pieces). So a row's result does not depend on
// its alignment or on the size of the batch. Rows 8,192 x dim 1,024, bf16 (84 MB): 14.2 us,
// 5.9 TB/s; the block per row below takes 18.1 us.
// ------------------------------------------------------------------------------------------
template <typename XT, typename GT, int N, int RES>
__global__ __launch_bounds__(256) void fl_gate_residual_norm_kernel(
    const XT* __restrict__ x, const GT* __restrict__ out, const GT* __restrict__ gpre,
    int64_t gstride, int64_t rows, int dim, const void* __restrict__ w, int w16, float eps,
    float inv_dim, XT* __restrict__ x_new, XT* __restrict__ normed) {
  constexpr int NV = RES / (64 * N);  // accesses per piece and lane
  extern __shared__ float s_rows[];
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= rows) return;  // whole waves; no barrier follows
  const int lane = threadIdx.x & 63;
  float* s_row = s_rows + (threadIdx.x >> 6) * RES;
  const int64_t base = row * dim;
  const GT* grow = gpre + row * gstride;
  float v[NV][N];
  auto residual = [&](int c, float* o) {
    float g[N], y[N], xx[N];
    Vec<GT, N>::load(grow + c, g);
    Vec<GT, N>::load(out + base + c, y);
    Vec<XT, N>::load(x + base + c, xx);
#pragma unroll
    for (int j = 0; j < N; ++j)
      o[j] = round_as<XT>(xx[j] + round_as<GT>(y[j] * round_as<GT>(sigmoid<GT>(g[j]))));
  };
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < dim; c0 += RES) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int o = (i * 64 + lane) * N, c = c0 + o;
#pragma unroll
      for (int j = 0; j < N; ++j) v[i][j] = 0.f;
      if (c < dim) residual(c, v[i]);
#pragma unroll
      for (int j = 0; j < N; ++j) s_row[o + j] = v[i][j];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // one wave's LDS operations complete in order
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = 0; i < RES / 256; ++i)
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float q = s_row[256 * i + 64 * k + lane];
        acc[k] = fmaf(q, q, acc[k]);
      }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  float tot = 0.f;
#pragma unroll
  for (int k = 0; k < 4; ++k) tot += wave_sum(acc[k]);
  const float scale = rsqrtf(fmaf(tot, inv_dim, eps));
  for (int c0 = 0; c0 < dim; c0 += RES) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = c0 + (i * 64 + lane) * N;
      if (c >= dim) continue;
      if (dim > RES) residual(c, v[i]);  // only the last piece is still held
      float ww[N], h[N];
      load_weight<N>(w, w16, c, ww);
#pragma unroll
      for (int j = 0; j < N; ++j) h[j] = (v[i][j] * scale) * ww[j];
      Vec<XT, N>::store(x_new + base + c, v[i]);
      Vec<XT, N>::store(normed + base + c, h);
    }
  }
}

// The same with a block of four waves per row, one element per thread and access: what a row without 16-byte
// access takes, where a wave alone would run through its elements four times as long (and through its two
// exponential chains twice, past one piece). NPER: elements that a thread keeps, 0 for longer rows, which are
// formed twice. The sum has the order above: thread c's chain is columns c, c + 256, ...
template <typename XT, typename GT, int NPER>
__global__ __launch_bounds__(256) void fl_gate_residual_norm_block_kernel(
    const XT* __restrict__ x, const GT* __restrict__ out, const GT* __restrict__ gpre, int64_t gstride, int dim,
    const void* __restrict__ w, int w16, float eps, float inv_dim, XT* __restrict__ x_new, XT* __restrict__ normed) {
  __shared__ float s_sum[4];
  const int64_t base = (int64_t)blockIdx.x * dim;
  const GT* grow = gpre + (int64_t)blockIdx.x * gstride;
  auto residual = [&](int c) {
    const float prod = round_as<GT>(load_as<GT>(out + base + c) * round_as<GT>(sigmoid<GT>(load_as<GT>(grow + c))));
    return round_as<XT>(load_as<XT>(x + base + c) + prod);
  };
  float v[NPER > 0 ? NPER : 1], acc = 0.f;
  if constexpr (NPER > 0) {
#pragma unroll
    for (int i = 0; i < NPER; ++i) {
      const int c = threadIdx.x + 256 * i;
      v[i] = c < dim ? residual(c) : 0.f;
      acc = fmaf(v[i], v[i], acc);
    }
  } else {
    for (int c = threadIdx.x; c < dim; c += 256) {
      const float r = residual(c);
      acc = fmaf(r, r, acc);
    }
  }
  acc = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) s_sum[threadIdx.x >> 6] = acc;
  __syncthreads();
  const float tot = ((s_sum[0] + s_sum[1]) + s_sum[2]) + s_sum[3], scale = rsqrtf(fmaf(tot, inv_dim, eps));
  auto put = [&](int c, float r, float weight) {
    store_as(x_new + base + c, r);
    store_as(normed + base + c, (r * scale) * weight);
  };
  if constexpr (NPER > 0) {
#pragma unroll
    for (int i = 0; i < NPER; ++i) {
      const int c = threadIdx.x + 256 * i;
      if (c >= dim) continue;
      float ww;
      load_weight<1>(w, w16, c, &ww);
      put(c, v[i], ww);
    }
  } else {
    auto again = [&](const auto* weight) {  // a branch on the weight's type per element cost 5 %
      for (int c = threadIdx.x; c < dim; c += 256) put(c, residual(c), load_as(weight + c));
    };
    if (w16) again(static_cast<const bf16_bits*>(w));
    else again(static_cast<const float*>(w));
  }
}

template <typename XT, typename GT>
int launch_gate_residual_norm(const void* x, const void* out, const void* gate_pre, int64_t rows,
                              int64_t dim, int64_t gate_stride, const void* w, int w16, float eps,
                              void* x_new, void* normed, hipStream_t s) {
  const float inv = (float)(1.0 / (double)dim);
#define FL_GRN1(N, RES)                                                                         \
  {                                                                                             \
    fl_gate_residual_norm_kernel<XT, GT, N, RES><<<(unsigned)cdiv(rows, 4), 256, 4 * RES * 4, s>>>( \
        static_cast<const XT*>(x), static_cast<const GT*>(out), static_cast<const GT*>(gate_pre), \
        gate_stride, rows, (int)dim, w, w16, eps, inv, static_cast<XT*>(x_new),                 \
        static_cast<XT*>(normed));                                                              \
    return hip_status(hipGetLastError());                                                       \
  }
#define FL_GRB(NPER)                                                                              \
  {                                                                                               \
    fl_gate_residual_norm_block_kernel<XT, GT, NPER><<<(unsigned)rows, 256, 0, s>>>(              \
        static_cast<const XT*>(x), static_cast<const GT*>(out), static_cast<const GT*>(gate_pre), \
        gate_stride, (int)dim, w, w16, eps, inv, static_cast<XT*>(x_new), static_cast<XT*>(normed)); \
    return hip_status(hipGetLastError());                                                         \
  }
  // 16-byte accesses: whole vectors per row and every row start aligned
  const bool vec = dim % 8 == 0 && gate_stride % 8 == 0 && aligned(x, 16) && aligned(out, 16) &&
                   aligned(gate_pre, 16) && aligned(w, 16) && aligned(x_new, 16) && aligned(normed, 16);
  // A wave per row and 16 bytes a lane pay once the rows are many enough to be bound by memory, and the
  // sooner the fewer bytes a row has; with few rows four waves finish a row sooner than one. us, wave | block:
  //   bf16 / bf16, dim 1,024:   64 rows 3.3 | 3.1,  1,000 4.2 | 4.0,  2,048 5.5 | 5.5,  4,096 8.6 | 9.8,  16,384 26 | 33
  //   fp32 / bf16, dim 1,024:   2,048 rows 8.2 | 6.6,  4,096 14.1 | 13.1,  8,192 23.7 | 23.1,  16,384 49 | 56
  //   fp32 / fp32, dim 1,024:   1,000 rows 5.7 | 4.7,  4,096 15.5 | 15.5,  16,384 66 | 65
  //   bf16 / bf16, dim 4,096:   64 rows 9.8 | 8.3,  1,000 14.0 | 15.2,  4,096 40 | 44
  //   256 and fewer columns:    bf16 8,192 rows 6.6 | 5.9,  16,384 11.2 | 12.0
  //   no 16-byte access, bf16, dim 1,022:  64 rows 8.5 | 3.2,  4,096 21 | 10.4,  16,384 49 | 35
  // (one row per block of the wave kernel instead of four: within 2 % from 512 rows on)
  if constexpr (sizeof(XT) == 2 || sizeof(GT) == 2) {
    if (vec && rows * dim >= (dim <= 256 ? 1 << 22 : sizeof(XT) == 2 ? 1 << 21 : 1 << 23)) {
      if (dim <= 512) FL_GRN1(8, 512)
      if (dim <= 1024) FL_GRN1(8, 1024)
      FL_GRN1(8, 2048)
    }
  }
  if (dim <= 256 && rows >= 16384) FL_GRN1(1, 256)
  if (dim <= 256) FL_GRB(1)
  if (dim <= 512) FL_GRB(2)
  if (dim <= 1024) FL_GRB(4)
  if (dim <= 2048) FL_GRB(8)
  FL_GRB(0)
#undef FL_GRB
#undef FL_GRN1
}

// ------------------------------------------------------------------------------------------
// out = silu(gate) * up with [gate | up] = the packed GEMM output, 3 * rows * hidden elements
// moved: bound by memory. 8 elements (16 bytes of bf16) per thread and access.
// Rows 8,192 x hidden 2,528, bf16 (124 MB): 22.9 us, 5.4 TB/s with part of it in the Infinity Cache;
// one element per thread with a 64-bit division for its row took 43.0 us.
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void fl_swiglu_vec_kernel(const T* __restrict__ gu, uint32_t n_vec,
                                                            uint32_t row_vecs, int hidden,
                                                            T* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= n_vec) return;
  const uint32_t r = i / row_vecs;
  const T* p = gu + (int64_t)r * hidden + (int64_t)i * 8;  // row r of 2 * hidden, column 8 * (i % row_vecs)
  float g[8], u[8], o[8];
  Vec<T, 8>::load(p, g);
  Vec<T, 8>::load(p + hidden, u);
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = round_as<T>(silu<T>(g[j])) * u[j];
  Vec<T, 8>::store(out + (int64_t)i * 8, o);
}

template <typename T>
__global__ __launch_bounds__(256) void fl_swiglu_kernel(const T* __restrict__ gu, int64_t rows,
                                                        int hidden, T* __restrict__ out) {
  const int64_t n = rows * hidden;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / hidden;
    const int j = (int)(i - r * hidden);
    const float g = load_as<T>(gu + r * 2 * hidden + j);
    const float u = load_as<T>(gu + r * 2 * hidden + hidden + j);
    store_as(out + i, round_as<T>(silu<T>(g)) * u);
  }
}

template <typename T>
int launch_swiglu(const void* gate_up, int64_t rows, int64_t hidden, void* out, hipStream_t s) {
  const T* gu = static_cast<const T*>(gate_up);
  T* o = static_cast<T*>(out);
  const int64_t n = rows * hidden;
  if (hidden % 8 == 0 && aligned(gate_up, 16) && aligned(out, 16) && n / 8 < ((int64_t)1 << 31)) {
    fl_swiglu_vec_kernel<T><<<(unsigned)cdiv(n / 8, 256), 256, 0, s>>>(gu, (uint32_t)(n / 8),
                                                                       (uint32_t)(hidden / 8), (int)hidden, o);
  } else {
    const unsigned blocks = (unsigned)(cdiv(n, 256) < 4096 ? cdiv(n, 256) : 4096);
    fl_swiglu_kernel<T><<<blocks, 256, 0, s>>>(gu, rows, (int)hidden, o);
  }
  return hip_status(hipGetLastError());
}

}  // namespace

extern "C" {

int fl_gate_residual_norm_w(const void* x, int x_dtype, const void* out, const void* gate_pre,
                            int g_dtype, int64_t rows, int64_t dim, int64_t gate_stride,
                            const void* norm_weight, int w_dtype, float eps, void* x_new,
                            void* normed, void* stream) {
  if (!dtype_ok(x_dtype) || !dtype_ok(g_dtype) || !dtype_ok(w_dtype)) return FL_ERR_DTYPE;
  if (rows <= 0 || dim <= 0 || rows > ((int64_t)1 << 31) - 1 || dim > ((int64_t)1 << 24))
    return FL_ERR_INVALID_ARGUMENT;
  if (gate_stride < dim || gate_stride > ((int64_t)1 << 31)) return FL_ERR_INVALID_ARGUMENT;
  if (!x || !out || !gate_pre || !norm_weight || !x_new || !normed || !(eps >= 0.f))
    return FL_ERR_INVALID_ARGUMENT;
  const size_t xs = esize(x_dtype), gs = esize(g_dtype);
  if (!aligned(x, xs) || !aligned(x_new, xs) || !aligned(normed, xs) || !aligned(out, gs) ||
      !aligned(gate_pre, gs) || !aligned(norm_weight, esize(w_dtype)))
    return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool x16 = x_dtype == FL_DTYPE_BF16, g16 = g_dtype == FL_DTYPE_BF16;
  const int w16 = w_dtype == FL_DTYPE_BF16;
#define FL_GRN(X, G) \
  return launch_gate_residual_norm<X, G>(x, out, gate_pre, rows, dim, gate_stride, norm_weight, w16, eps, x_new, normed, s);
  if (x16 && g16) { FL_GRN(bf16_bits, bf16_bits) }
  if (x16) { FL_GRN(bf16_bits, float) }
  if (g16) { FL_GRN(float, bf16_bits) }
  FL_GRN(float, float)
#undef FL_GRN
}

int fl_gate_residual_norm(const void* x, int x_dtype, const void* out, const void* gate_pre,
                          int g_dtype, int64_t rows, int64_t dim, int64_t gate_stride,
                          const float* norm_weight, float eps, void* x_new, void* normed,
                          void* stream) {
  return fl_gate_residual_norm_w(x, x_dtype, out, gate_pre, g_dtype, rows, dim, gate_stride,
                                 norm_weight, FL_DTYPE_F32, eps, x_new, normed, stream);
}

int fl_swiglu(const void* gate_up, int dtype, int64_t rows, int64_t hidden, void* out,
              void* stream) {
  if (!dtype_ok(dtype)) return FL_ERR_DTYPE;
  if (rows <= 0 || hidden <= 0 || hidden > ((int64_t)1 << 30)) return FL_ERR_INVALID_ARGUMENT;
  if (!gate_up || !out) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(gate_up, esize(dtype)) || !aligned(out, esize(dtype))) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return dtype == FL_DTYPE_BF16 ? launch_swiglu<bf16_bits>(gate_up, rows, hidden, out, s)
                                : launch_swiglu<float>(gate_up, rows, hidden, out, s);
}

}  // extern "C"
