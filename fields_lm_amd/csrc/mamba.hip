// mamba.hip — the Mamba-2 mixer between its two projections (no gradient needed): causal depthwise
// convolution, softplus, the state-space scan, the D skip and the gated RMSNorm, for a whole
// sequence (fl_mamba_prefill) and for one token (fl_mamba_step). The mixer's maths and parameter
// layout are those of the model's Mamba-2 blocks (reference: src/fields_official/reference/
// official_source/field_fusion_wiki100_mamba2_v25.py:73-91, 455-468); the scan is the chunked
// state-space-duality form (Dao & Gu, 2024):
//   h_t = exp(dt_t A) h_{t-1} + dt_t x_t B_t^T,   y_t = h_t C_t + D x_t       (per head)
// with 64 channels per head, 128 states and one B / C group.
//
// Every product is fp32 (v_mfma_f32_16x16x4_f32): x, B, C, the decays and the state are fp32 in the
// stock path, and they stay so.
#include "fl_common.h"

namespace {

using namespace fl;

constexpr int kQ = 64;      // tokens per chunk: one per lane in the decay scan
constexpr int kP = 64;      // channels per head
constexpr int kN = 128;     // states
constexpr int kTaps = 4;    // convolution width
constexpr float kLn2 = 0.6931471805599453f;
constexpr int kXStride = 68;   // floats per staged x row: 4 banks further per row, so that 16 lanes'
constexpr int kHStride = 132;  // 16-byte reads of 16 rows take every bank once (state rows alike)
// Operand fragments, as the scan's lanes read them: 16 bytes per lane, a wave's 1 KB contiguous.
// C: [row tile 4][k block 8], B transposed: [state tile 8][k block 4], C B^T: [row tile 4][k block 4]
constexpr int kCFrag = 4 * 8 * 256, kBFrag = 8 * 4 * 256, kGFrag = 4 * 4 * 256;
constexpr int kChunkFrags = kCFrag + kBFrag + kGFrag;  // floats per (sequence, chunk): 80 KB

__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// F.softplus: the identity above its threshold of 20
__device__ __forceinline__ float softplus(float x) { return x > 20.0f ? x : log1pf(expf(x)); }

template <typename T>
__device__ __forceinline__ void load_pair(const T* p, float* o);
template <>
__device__ __forceinline__ void load_pair<float>(const float* p, float* o) {
  const f32x2 v = *reinterpret_cast<const f32x2*>(p);
  o[0] = v.x; o[1] = v.y;
}
template <>
__device__ __forceinline__ void load_pair<bf16_bits>(const bf16_bits* p, float* o) {
  const uint32_t w = *reinterpret_cast<const uint32_t*>(p);
  o[0] = bf16_lo(w); o[1] = bf16_hi(w);
}

// a pair at byte offset vo (lane) + so (wave), 0 past the buffer
template <typename T>
__device__ __forceinline__ void load_pair(rsrc_t r, int vo, int so, float* o);
template <>
__device__ __forceinline__ void load_pair<float>(rsrc_t r, int vo, int so, float* o) {
  const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(r, vo, so, 0);
  o[0] = __uint_as_float(w.x); o[1] = __uint_as_float(w.y);
}
template <>
__device__ __forceinline__ void load_pair<bf16_bits>(rsrc_t r, int vo, int so, float* o) {
  const uint32_t w = __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0);
  o[0] = bf16_lo(w); o[1] = bf16_hi(w);
}

struct ConvParams {  // depthwise weights [channels, 4] and bias [channels], one type for both
  const void* w;
  const void* b;
  int is16;
  __device__ __forceinline__ void get(int c, float* wt, float& bias) const {
    if (is16) {
      for (int k = 0; k < kTaps; ++k) wt[k] = load_as<bf16_bits>(static_cast<const bf16_bits*>(w) + kTaps * c + k);
      bias = load_as<bf16_bits>(static_cast<const bf16_bits*>(b) + c);
    } else {
      for (int k = 0; k < kTaps; ++k) wt[k] = static_cast<const float*>(w)[kTaps * c + k];
      bias = static_cast<const float*>(b)[c];
    }
  }
};

// out[t] = silu(bias + sum_k w[k] in[t - 3 + k]), the taps added in the stock order
__device__ __forceinline__ float conv_silu(const float* wt, float bias, float a, float b, float c, float d) {
  float v = fmaf(a, wt[0], bias);
  v = fmaf(b, wt[1], v);
  v = fmaf(c, wt[2], v);
  return silu_precise<false>(fmaf(d, wt[3], v));
}

// ------------------------------------------------------------------------------------------
// Per (sequence, chunk): B and C after their convolution, C B^T, and dt after softplus, written in
// the scan's operand order. One block of 16 waves; the [64 x 64] product is one tile per wave.
// Rows at and past L are zero (dt 0: decay 1, no input).
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(1024) void fl_mamba_chunk_kernel(
    const T* __restrict__ xbc, const T* __restrict__ dt_raw, int64_t sb, int64_t st, int L, int H,
    int n_chunks, ConvParams conv, const float* __restrict__ dt_bias, float* __restrict__ frags,
    float* __restrict__ dt_out) {
  __shared__ float s_b[kQ * kHStride], s_c[kQ * kHStride];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6);
  const int b = blockIdx.x / n_chunks, chunk = blockIdx.x - b * n_chunks, t0 = chunk * kQ;
  const int inner = H * kP;
  {
    const int c = tid & 255, g = tid >> 8;  // channel inner + c, 16 rows from t0 + 16 g
    float wt[kTaps], bias, in[kTaps + 15];
    conv.get(inner + c, wt, bias);
    const T* p = xbc + b * sb + inner + c;
#pragma unroll
    for (int i = 0; i < kTaps + 15; ++i) in[i] = load_as<T>(p + (int64_t)min(max(t0 + 16 * g - 3 + i, 0), L - 1) * st);
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (t0 + 16 * g - 3 + i < 0) in[i] = 0.f;
    float* dst = (c < kN ? s_b + c : s_c + c - kN) + 16 * g * kHStride;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float v = conv_silu(wt, bias, in[i], in[i + 1], in[i + 2], in[i + 3]);
      dst[i * kHStride] = t0 + 16 * g + i < L ? v : 0.f;
    }
  }
  for (int i = tid; i < kQ * H; i += 1024) {
    const int t = i / H, h = i - t * H;
    const float v = t0 + t < L ? softplus(load_as<T>(dt_raw + b * sb + (int64_t)(t0 + t) * st + h) + dt_bias[h]) : 0.f;
    dt_out[((int64_t)b * H + h) * (n_chunks * kQ) + t0 + t] = v;
  }
  __syncthreads();
  float* f = frags + (int64_t)blockIdx.x * kChunkFrags + 4 * lane;
  const int r = lane & 15, k4 = 4 * (lane >> 4);
  {  // C B^T, tile (rows 16 (wave / 4), columns 16 (wave % 4)): rows of the result are B's tokens
    const int tt = wave >> 2, j = wave & 3;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int n = 0; n < kN; n += 16) {
      const f32x4 a = *reinterpret_cast<const f32x4*>(s_b + (16 * j + r) * kHStride + n + k4);
      const f32x4 c = *reinterpret_cast<const f32x4*>(s_c + (16 * tt + r) * kHStride + n + k4);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc = mfma4(a[i], c[i], acc);
    }
    *reinterpret_cast<f32x4*>(f + kCFrag + kBFrag + (tt * 4 + j) * 256) = acc;
  }
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int id = wave * 2 + q;  // 32 fragments of each
    *reinterpret_cast<f32x4*>(f + id * 256) =
        *reinterpret_cast<const f32x4*>(s_c + (16 * (id >> 3) + r) * kHStride + 16 * (id & 7) + k4);
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = s_b[(16 * (id & 3) + k4 + i) * kHStride + 16 * (id >> 2) + r];
    *reinterpret_cast<f32x4*>(f + kCFrag + id * 256) = v;
  }
}

// ------------------------------------------------------------------------------------------
// The scan: one block per (sequence, head, PT x 16 of its 64 channels) walks the chunks in order
// with its state [16 PT x 128] in accumulators, so no chunk state ever reaches memory. Per chunk
//   waves 0-3:  y = exp(acs_t) C h^T + (C B^T o exp(acs_t - acs_s) dt_s) x + D x    (16 rows each)
//   waves 4-7:  h = exp(acs_end) h + (x exp(acs_end - acs_s) dt_s)^T B          (32 states each)
// with acs the running sum of dt A within the chunk, in log2 units (each decay is one v_exp_f32),
// summed in double and kept as two floats: a decay is the exponential of the difference of two sums
// that may be large, and rounded sums cost 5e-6 of a fast-decaying head's state against 8e-7 stock.
// Bound by the fp32 matrix rate: 10.7 GFLOP at 8,192 tokens x 32 heads, 68 us at 157 TFLOP/s. The
// C, B and C B^T operands are no other wave's, so they come from L2 straight into registers, one
// chunk ahead; only x (all waves) and h (produced by state, consumed by row) pass through LDS. The
// two roles need the state before the chunk only, so they run side by side, two waves per SIMD, one's
// exponentials and convolution under the other's products.
// Work items of one sequence sit on neighbouring XCDs' L2s (contiguous work per XCD).
// 4 x 2,048 tokens, 32 heads: 145 us, 74 TFLOP/s (whole mixer between its projections 182 us, where
// the stock ops' 75 launches took 1,690 us).
// ------------------------------------------------------------------------------------------
template <typename T, int PT>
__global__ __launch_bounds__(512, 2) void fl_mamba_scan_kernel(
    const T* __restrict__ xbc, int64_t sb, int64_t st, int L, int H, int n_chunks, ConvParams conv,
    const float* __restrict__ A_log, const float* __restrict__ D, const float* __restrict__ frags,
    const float* __restrict__ dt_sp, float* __restrict__ y, float* __restrict__ ssm_out) {
  constexpr int PB = 16 * PT;                     // channels of this block
  constexpr int kPairs = PB / 2, kRows = 64 * kPairs / 512;  // conv: channel pair x kRows tokens per thread
  constexpr int NS = kP / PB;
  __shared__ float s_x[2][PB * kXStride], s_h[2][PB * kHStride], s_acs[2][kQ], s_lo[2][kQ], s_dt[2][kQ];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), role = wave >> 2, w4 = wave & 3;
  const int r = lane & 15, k4 = 4 * (lane >> 4);
  // blocks go to XCD blockIdx % 8: give each XCD a contiguous run of work items
  int work = blockIdx.x;
  if ((gridDim.x & 7) == 0) work = (work & 7) * (gridDim.x >> 3) + (work >> 3);
  const int split = work % NS, h = (work / NS) % H, b = work / (NS * H);
  const int inner = H * kP, ch0 = h * kP + split * PB;
  const double a2 = -(double)expf(A_log[h]) * 1.4426950408889634;
  const float d_skip = D[h];

  const int cp = tid % kPairs, tg = tid / kPairs;
  float wt[2][kTaps], bias[2];
  conv.get(ch0 + 2 * cp, wt[0], bias[0]);
  conv.get(ch0 + 2 * cp + 1, wt[1], bias[1]);
  const T* xp = xbc + b * sb + ch0 + 2 * cp;
  const float* fbase = frags + (int64_t)b * n_chunks * kChunkFrags + 4 * lane;
  const float* dtp = dt_sp + ((int64_t)b * H + h) * (n_chunks * kQ) + lane;

  float raw[kRows + 3][2], dt;
  // rows 64 chunk - 3 .. of a later chunk (chunk < n_chunks) through a buffer that ends with the
  // sequence: no branch per row, whose loads cost 57 us of 178 at 4 x 2,048 tokens
  const int row_bytes = (int)(st * sizeof(T)), x_off = tg * kRows * row_bytes + 2 * cp * (int)sizeof(T);
  auto fetch_x = [&](int chunk) {
    const int first = chunk * kQ - 3, rows = min(L - first, kQ + 3);
    const rsrc_t rs = make_rsrc(xbc + b * sb + ch0 + (int64_t)first * st, (uint32_t)(rows * row_bytes));
#pragma unroll
    for (int i = 0; i < kRows + 3; ++i) load_pair<T>(rs, x_off, i * row_bytes, raw[i]);
    dt = dtp[chunk * kQ];
  };
  // x of a fetched chunk, channel-major, and its decays (one wave) into the buffers `buf`
  auto stage = [&](int buf) {
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      float* dst = &s_x[buf][(2 * cp + e) * kXStride + tg * kRows];
#pragma unroll
      for (int i = 0; i < kRows; ++i)
        dst[i] = conv_silu(wt[e], bias[e], raw[i][e], raw[i + 1][e], raw[i + 2][e], raw[i + 3][e]);
    }
    if (wave == 4) {
      double s = dt * a2;
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        const double o = __shfl_up(s, m);
        if (lane >= m) s += o;
      }
      const float hi = (float)s;
      s_acs[buf][lane] = hi;
      s_lo[buf][lane] = (float)(s - hi);
      s_dt[buf][lane] = dt;
    }
  };
  // role 0: C (32 floats per lane) and C B^T (16); role 1: B (32)
  f32x4 f1[8], f2[4];
  auto fetch_f1 = [&](int chunk) {
    const float* f = fbase + (int64_t)chunk * kChunkFrags + role * kCFrag + w4 * 8 * 256;
#pragma unroll
    for (int j = 0; j < 8; ++j) f1[j] = *reinterpret_cast<const f32x4*>(f + j * 256);
  };
  auto fetch_f2 = [&](int chunk) {
    const float* f = fbase + (int64_t)chunk * kChunkFrags + kCFrag + kBFrag + w4 * 4 * 256;
#pragma unroll
    for (int j = 0; j < 4; ++j) f2[j] = *reinterpret_cast<const f32x4*>(f + j * 256);
  };
#pragma unroll
  for (int i = 0; i < kRows + 3; ++i) {  // chunk 0: the rows before the sequence are zero
    const int t = tg * kRows - 3 + i;
    raw[i][0] = raw[i][1] = 0.f;
    if (t >= 0 && t < L) load_pair<T>(xp + (int64_t)t * st, raw[i]);
  }
  dt = dtp[0];
  fetch_f1(0);
  if (role == 0) fetch_f2(0);
  f32x4 hacc[2][PT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int p = 0; p < PT; ++p) hacc[q][p] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int i = tid; i < PB * kHStride; i += 512) s_h[0][i] = 0.f;
  stage(0);
  if (n_chunks > 1) fetch_x(1);

  for (int chunk = 0; chunk < n_chunks; ++chunk) {
    const int buf = chunk & 1;
    const int next = chunk + 1 < n_chunks ? chunk + 1 : chunk;
    // The one barrier of a chunk: its x, decays and entering state are visible after it, and every
    // reader of the other buffers, which this chunk's end writes, has passed it.
    __syncthreads();
    f32x4 xf[PT][4];
#pragma unroll
    for (int p = 0; p < PT; ++p)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xf[p][j] = *reinterpret_cast<const f32x4*>(&s_x[buf][(16 * p + r) * kXStride + 16 * j + k4]);
    if (role == 0) {
      const int tl = 16 * w4 + r;  // this lane's row of the chunk
      const float acs_t = s_acs[buf][tl], lo_t = s_lo[buf][tl];
      f32x4 acc[PT];
#pragma unroll
      for (int p = 0; p < PT; ++p) acc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        f32x4 hf[PT];
#pragma unroll
        for (int p = 0; p < PT; ++p)
          hf[p] = *reinterpret_cast<const f32x4*>(&s_h[buf][(16 * p + r) * kHStride + 16 * j + k4]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int p = 0; p < PT; ++p) acc[p] = mfma4(hf[p][i], f1[j][i], acc[p]);
      }
      fetch_f1(next);
      const float et = __builtin_amdgcn_exp2f(acs_t) * fmaf(lo_t, kLn2, 1.0f);
#pragma unroll
      for (int p = 0; p < PT; ++p) acc[p] *= et;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (j <= w4) {  // causal: later row tiles see nothing of this column tile
          const f32x4 as = *reinterpret_cast<const f32x4*>(&s_acs[buf][16 * j + k4]);
          const f32x4 ls = *reinterpret_cast<const f32x4*>(&s_lo[buf][16 * j + k4]);
          const f32x4 ds = *reinterpret_cast<const f32x4*>(&s_dt[buf][16 * j + k4]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float decay = __builtin_amdgcn_exp2f((acs_t - as[i]) + (lo_t - ls[i]));
            const float m = 16 * j + k4 + i <= tl ? f2[j][i] * (decay * ds[i]) : 0.f;
#pragma unroll
            for (int p = 0; p < PT; ++p) acc[p] = mfma4(xf[p][j][i], m, acc[p]);
          }
        }
      }
      fetch_f2(next);
      const int t = chunk * kQ + tl;
      if (t < L) {
        float* yo = y + ((int64_t)b * L + t) * inner + ch0 + k4;
#pragma unroll
        for (int p = 0; p < PT; ++p) {
          f32x4 o = acc[p];
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = fmaf(d_skip, s_x[buf][(16 * p + k4 + i) * kXStride + tl], o[i]);
          *reinterpret_cast<f32x4*>(yo + 16 * p) = o;
        }
      }
    } else {
      const float acs_end = s_acs[buf][kQ - 1], lo_end = s_lo[buf][kQ - 1];
      const float ee = __builtin_amdgcn_exp2f(acs_end) * fmaf(lo_end, kLn2, 1.0f);
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int p = 0; p < PT; ++p) hacc[q][p] *= ee;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 as = *reinterpret_cast<const f32x4*>(&s_acs[buf][16 * j + k4]);
        const f32x4 ls = *reinterpret_cast<const f32x4*>(&s_lo[buf][16 * j + k4]);
        const f32x4 ds = *reinterpret_cast<const f32x4*>(&s_dt[buf][16 * j + k4]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float wk = __builtin_amdgcn_exp2f((acs_end - as[i]) + (lo_end - ls[i])) * ds[i];
#pragma unroll
          for (int p = 0; p < PT; ++p) {
            const float xw = xf[p][j][i] * wk;
#pragma unroll
            for (int q = 0; q < 2; ++q) hacc[q][p] = mfma4(f1[4 * q + j][i], xw, hacc[q][p]);
          }
        }
      }
      fetch_f1(next);
    }
    if (chunk + 1 < n_chunks) {
      stage(buf ^ 1);
      fetch_x(chunk + 2 < n_chunks ? chunk + 2 : next);  // (the last ones again: unused)
      if (role == 1) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int p = 0; p < PT; ++p)
            *reinterpret_cast<f32x4*>(&s_h[buf ^ 1][(16 * p + r) * kHStride + 32 * w4 + 16 * q + k4]) = hacc[q][p];
      }
    }
  }
  if (ssm_out != nullptr && role == 1) {
    float* so = ssm_out + (((int64_t)b * H + h) * kP + split * PB + r) * kN + 32 * w4 + k4;
#pragma unroll
    for (int q = 0; q < 2; ++q)
#pragma unroll
      for (int p = 0; p < PT; ++p) *reinterpret_cast<f32x4*>(so + 16 * p * kN + 16 * q) = hacc[q][p];
  }
}

// ------------------------------------------------------------------------------------------
// Gated RMSNorm over the whole inner width: v = y silu(z), out = (v rsqrt(mean v^2 + eps)) w, fp32
// maths, one wave per row. Bound by memory: y fp32 and z in, out once.
// ------------------------------------------------------------------------------------------
template <typename T, typename OT, int N, int NV>
__global__ __launch_bounds__(256) void fl_gated_norm_kernel(
    const float* __restrict__ y, const T* __restrict__ z, int64_t zsb, int64_t zst, int64_t rows,
    int L, int dim, const void* __restrict__ w, int w16, float eps, float inv_dim, OT* __restrict__ out) {
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const int64_t b = row / L;
  const T* zr = z + b * zsb + (row - b * L) * zst;
  const float* yr = y + row * dim;
  OT* o = out + row * dim;
  auto value = [&](int c, float* v) {
    float g[N];
    Vec<float, N>::load(yr + c, v);
    Vec<T, N>::load(zr + c, g);
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] *= silu_precise<false>(g[j]);
  };
  auto finish = [&](int c, const float* v, float scale) {
    float ww[N], q[N];
    if (w16) Vec<bf16_bits, N>::load(static_cast<const bf16_bits*>(w) + c, ww);
    else Vec<float, N>::load(static_cast<const float*>(w) + c, ww);
#pragma unroll
    for (int j = 0; j < N; ++j) q[j] = (v[j] * scale) * ww[j];
    Vec<OT, N>::store(o + c, q);
  };
  float acc = 0.f;
  if constexpr (NV > 0) {
    float v[NV][N];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = (i * 64 + lane) * N;
      if (c < dim) {
        value(c, v[i]);
#pragma unroll
        for (int j = 0; j < N; ++j) acc = fmaf(v[i][j], v[i][j], acc);
      }
    }
    const float scale = rsqrtf(fmaf(wave_sum(acc), inv_dim, eps));
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = (i * 64 + lane) * N;
      if (c < dim) finish(c, v[i], scale);
    }
  } else {
    for (int c = lane * N; c < dim; c += 64 * N) {
      float v[N];
      value(c, v);
#pragma unroll
      for (int j = 0; j < N; ++j) acc = fmaf(v[j], v[j], acc);
    }
    const float scale = rsqrtf(fmaf(wave_sum(acc), inv_dim, eps));
    for (int c = lane * N; c < dim; c += 64 * N) {
      float v[N];
      value(c, v);
      finish(c, v, scale);
    }
  }
}

template <typename T, typename OT>
int launch_gated_norm(const float* y, const T* z, int64_t zsb, int64_t zst, int64_t rows, int L, int dim,
                      const void* w, int w16, float eps, OT* out, hipStream_t s) {
  // one row per block while the rows are few; whole call, one | four rows a block: 64 x 64 tokens 136.0 | 135.4 us,
  // 64 x 1 107.1 | 107.3, 8 x 64 33.1 | 33.5
  const unsigned waves = rows >= 4096 ? 4 : 1;
  const unsigned blocks = (unsigned)cdiv(rows, waves);
  const float inv = (float)(1.0 / (double)dim);
#define FL_GN(N, NV)                                                                              \
  {                                                                                               \
    fl_gated_norm_kernel<T, OT, N, NV><<<blocks, waves * 64, 0, s>>>(y, z, zsb, zst, rows, L, dim, w, \
                                                                      w16, eps, inv, out);        \
    return hip_status(hipGetLastError());                                                         \
  }
  const bool vec = dim % 8 == 0 && zst % 8 == 0 && zsb % 8 == 0 && aligned(z, 16) && aligned(out, 16) &&
                   aligned(w, 16);
  if (vec && dim <= 2048) FL_GN(8, 4)
  if (vec) FL_GN(8, 0)
  FL_GN(1, 0)
#undef FL_GN
}

// ------------------------------------------------------------------------------------------
// One token. Convolution: the window [B, channels, 4] shifts in place. State: one block per
// (sequence, head), the [64 x 128] state read and written once (16 bytes per lane, a wave two rows
// of 512 bytes), bound by that traffic: B=64, 32 heads 134 MB in 25.8 us,
// 5.2 TB/s (the stock ops of one token: 270 us in a graph, 48 us now).
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void fl_mamba_conv_step_kernel(const T* __restrict__ xbc, int64_t sb,
                                                                 int channels, ConvParams conv,
                                                                 float* __restrict__ window,
                                                                 float* __restrict__ xbc_out) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int64_t b = blockIdx.y;
  if (c >= channels) return;
  float wt[kTaps], bias;
  conv.get(c, wt, bias);
  f32x4* win = reinterpret_cast<f32x4*>(window + (b * channels + c) * kTaps);
  const f32x4 o = *win;
  const float in = load_as<T>(xbc + b * sb + c);
  *win = f32x4{o[1], o[2], o[3], in};
  xbc_out[b * channels + c] = conv_silu(wt, bias, o[1], o[2], o[3], in);
}

template <typename T>
__global__ __launch_bounds__(256) void fl_mamba_state_step_kernel(
    const float* __restrict__ xbc, const T* __restrict__ dt_raw, int64_t sb, int H,
    const float* __restrict__ dt_bias, const float* __restrict__ A_log, const float* __restrict__ D,
    float* __restrict__ ssm, float* __restrict__ y) {
  const int h = blockIdx.x, lane32 = threadIdx.x & 31, row = threadIdx.x >> 5;
  const int64_t b = blockIdx.y;
  const int channels = H * kP + 2 * kN;
  const float dt = softplus(load_as<T>(dt_raw + b * sb + h) + dt_bias[h]);
  const float decay = expf(dt * -expf(A_log[h])), d_skip = D[h];
  const float* xb = xbc + b * channels;
  const f32x4 bm = *reinterpret_cast<const f32x4*>(xb + H * kP + 4 * lane32);
  const f32x4 cm = *reinterpret_cast<const f32x4*>(xb + H * kP + kN + 4 * lane32);
  f32x4* s = reinterpret_cast<f32x4*>(ssm + ((b * H + h) * kP + row) * kN) + lane32;
  f32x4 v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = s[i * 8 * (kN / 4)];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x = xb[h * kP + row + 8 * i], xdt = x * dt;
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[i][j] = fmaf(xdt, bm[j], v[i][j] * decay);
      acc = fmaf(v[i][j], cm[j], acc);
    }
    s[i * 8 * (kN / 4)] = v[i];
#pragma unroll
    for (int m = 1; m < 32; m <<= 1) acc += __shfl_xor(acc, m);
    if (lane32 == 0) y[(b * H + h) * kP + row + 8 * i] = fmaf(d_skip, x, acc);
  }
}

struct MambaLayout {
  int64_t n_chunks;
  size_t frag_off, dt_off, y_off, bytes;
};

MambaLayout mamba_layout(int64_t B, int64_t L, int64_t H) {
  MambaLayout m;
  m.n_chunks = cdiv(L, kQ);
  m.frag_off = 0;
  m.dt_off = (size_t)(B * m.n_chunks) * kChunkFrags * 4;
  m.y_off = m.dt_off + (size_t)cdiv(B * H * m.n_chunks * kQ * 4, 256) * 256;
  m.bytes = m.y_off + (size_t)(B * L * H * kP) * 4;
  return m;
}

size_t mamba_step_bytes(int64_t B, int64_t H) {
  return (size_t)B * (H * kP + 2 * kN + H * kP) * 4;
}

bool mamba_args_ok(int dtype, int conv_dtype, int norm_dtype, int out_dtype, int* code) {
  *code = FL_ERR_DTYPE;
  return dtype_ok(dtype) && dtype_ok(conv_dtype) && dtype_ok(norm_dtype) && dtype_ok(out_dtype);
}

template <typename T>
int prefill_impl(const T* zx, int64_t B, int64_t L, int64_t H, int64_t sb, int64_t st, ConvParams conv,
                 const float* A_log, const float* dt_bias, const float* D, const void* norm_w, int nw16,
                 float eps, void* out, int out16, float* ssm_out, char* ws, hipStream_t s) {
  const MambaLayout m = mamba_layout(B, L, H);
  const int inner = (int)H * kP;
  const T* xbc = zx + inner;
  const T* dt_raw = xbc + inner + 2 * kN;
  float* frags = reinterpret_cast<float*>(ws + m.frag_off);
  float* dts = reinterpret_cast<float*>(ws + m.dt_off);
  float* y = reinterpret_cast<float*>(ws + m.y_off);
  const int nc = (int)m.n_chunks;
  fl_mamba_chunk_kernel<T><<<(unsigned)(B * nc), 1024, 0, s>>>(xbc, dt_raw, sb, st, (int)L, (int)H, nc, conv,
                                                               dt_bias, frags, dts);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_status(e);
  // A block takes 32 channels of a head once blocks of 16 would be more than the 256 CUs (they share less
  // of C, B and C B^T). us, 16 | 32 channels, 32 heads: 1 x 2,048 tokens 114 | 155, 2 x 1,024 73 | 94,
  // 3 x 1,024 120 | 98, 4 x 1,024 123 | 102, 8 x 1,024 222 | 182
  if (B * H * 4 > 256) {
    fl_mamba_scan_kernel<T, 2><<<(unsigned)(B * H * 2), 512, 0, s>>>(xbc, sb, st, (int)L, (int)H, nc, conv, A_log,
                                                                     D, frags, dts, y, ssm_out);
  } else {
    fl_mamba_scan_kernel<T, 1><<<(unsigned)(B * H * 4), 512, 0, s>>>(xbc, sb, st, (int)L, (int)H, nc, conv, A_log,
                                                                     D, frags, dts, y, ssm_out);
  }
  e = hipGetLastError();
  if (e != hipSuccess) return hip_status(e);
  return out16 ? launch_gated_norm<T, bf16_bits>(y, zx, sb, st, B * L, (int)L, inner, norm_w, nw16, eps,
                                                 static_cast<bf16_bits*>(out), s)
               : launch_gated_norm<T, float>(y, zx, sb, st, B * L, (int)L, inner, norm_w, nw16, eps,
                                             static_cast<float*>(out), s);
}

template <typename T>
int step_impl(const T* zx, int64_t B, int64_t H, int64_t sb, ConvParams conv, const float* A_log,
              const float* dt_bias, const float* D, const void* norm_w, int nw16, float eps, float* window,
              float* ssm, void* out, int out16, char* ws, hipStream_t s) {
  const int inner = (int)H * kP, channels = inner + 2 * kN;
  const T* xbc = zx + inner;
  const T* dt_raw = xbc + channels;
  float* xo = reinterpret_cast<float*>(ws);
  float* y = xo + B * channels;
  fl_mamba_conv_step_kernel<T><<<dim3((unsigned)cdiv(channels, 256), (unsigned)B), 256, 0, s>>>(
      xbc, sb, channels, conv, window, xo);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_status(e);
  fl_mamba_state_step_kernel<T><<<dim3((unsigned)H, (unsigned)B), 256, 0, s>>>(xo, dt_raw, sb, (int)H, dt_bias,
                                                                               A_log, D, ssm, y);
  e = hipGetLastError();
  if (e != hipSuccess) return hip_status(e);
  return out16 ? launch_gated_norm<T, bf16_bits>(y, zx, sb, sb, B, 1, inner, norm_w, nw16, eps,
                                                 static_cast<bf16_bits*>(out), s)
               : launch_gated_norm<T, float>(y, zx, sb, sb, B, 1, inner, norm_w, nw16, eps,
                                             static_cast<float*>(out), s);
}

}  // namespace

extern "C" {

size_t fl_mamba_workspace_bytes(int64_t B, int64_t L, int64_t heads) {
  if (B <= 0 || L <= 0 || heads <= 0) return 0;
  const size_t a = mamba_layout(B, L, heads).bytes, c = mamba_step_bytes(B, heads);
  return a > c ? a : c;
}

int fl_mamba_prefill(const void* zxbcdt, int dtype, int64_t B, int64_t L, int64_t heads, int64_t stride_b,
                     int64_t stride_t, const void* conv_w, const void* conv_b, int conv_dtype,
                     const float* A_log, const float* dt_bias, const float* D, const void* norm_w,
                     int norm_dtype, float eps, void* out, int out_dtype, float* ssm_out, void* workspace,
                     size_t workspace_bytes, void* stream) {
  int code;
  if (!mamba_args_ok(dtype, conv_dtype, norm_dtype, out_dtype, &code)) return code;
  if (B <= 0 || L <= 0 || heads <= 0 || heads > 1024 || B > 65535 || L > ((int64_t)1 << 26) ||
      B * heads > ((int64_t)1 << 20) || B * cdiv(L, kQ) > ((int64_t)1 << 30))
    return FL_ERR_INVALID_ARGUMENT;
  const int64_t width = 2 * heads * kP + 2 * kN + heads;
  if (stride_t < width || stride_b < 0 || (B > 1 && stride_b < (L - 1) * stride_t + width))
    return FL_ERR_INVALID_ARGUMENT;
  if (!zxbcdt || !conv_w || !conv_b || !A_log || !dt_bias || !D || !norm_w || !out || !(eps >= 0.f))
    return FL_ERR_INVALID_ARGUMENT;
  // channel pairs are read in one access; a chunk's rows lie within a buffer's 2 GiB
  if (stride_t > ((int64_t)1 << 22)) return FL_ERR_INVALID_ARGUMENT;
  if (stride_t % 2 || stride_b % 2 || !aligned(zxbcdt, 2 * esize(dtype))) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(conv_w, esize(conv_dtype)) || !aligned(conv_b, esize(conv_dtype)) || !aligned(A_log, 4) ||
      !aligned(dt_bias, 4) || !aligned(D, 4) || !aligned(norm_w, esize(norm_dtype)) ||
      !aligned(out, esize(out_dtype)) || !aligned(ssm_out, 16))
    return FL_ERR_INVALID_ARGUMENT;
  if (!workspace || workspace_bytes < mamba_layout(B, L, heads).bytes) return FL_ERR_WORKSPACE;
  if (!aligned(workspace, 16)) return FL_ERR_INVALID_ARGUMENT;
  const ConvParams conv{conv_w, conv_b, conv_dtype == FL_DTYPE_BF16};
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const int nw16 = norm_dtype == FL_DTYPE_BF16, o16 = out_dtype == FL_DTYPE_BF16;
  return dtype == FL_DTYPE_BF16
             ? prefill_impl(static_cast<const bf16_bits*>(zxbcdt), B, L, heads, stride_b, stride_t, conv, A_log,
                            dt_bias, D, norm_w, nw16, eps, out, o16, ssm_out, ws, s)
             : prefill_impl(static_cast<const float*>(zxbcdt), B, L, heads, stride_b, stride_t, conv, A_log,
                            dt_bias, D, norm_w, nw16, eps, out, o16, ssm_out, ws, s);
}

int fl_mamba_step(const void* zxbcdt, int dtype, int64_t B, int64_t heads, int64_t stride_b,
                  const void* conv_w, const void* conv_b, int conv_dtype, const float* A_log,
                  const float* dt_bias, const float* D, const void* norm_w, int norm_dtype, float eps,
                  float* conv_state, float* ssm, void* out, int out_dtype, void* workspace,
                  size_t workspace_bytes, void* stream) {
  int code;
  if (!mamba_args_ok(dtype, conv_dtype, norm_dtype, out_dtype, &code)) return code;
  if (B <= 0 || heads <= 0 || heads > 1024 || B > 65535) return FL_ERR_INVALID_ARGUMENT;
  if (stride_b < 2 * heads * kP + 2 * kN + heads) return FL_ERR_INVALID_ARGUMENT;
  if (!zxbcdt || !conv_w || !conv_b || !A_log || !dt_bias || !D || !norm_w || !out || !conv_state || !ssm ||
      !(eps >= 0.f))
    return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(zxbcdt, esize(dtype)) || !aligned(conv_w, esize(conv_dtype)) ||
      !aligned(conv_b, esize(conv_dtype)) || !aligned(A_log, 4) || !aligned(dt_bias, 4) || !aligned(D, 4) ||
      !aligned(norm_w, esize(norm_dtype)) || !aligned(out, esize(out_dtype)) || !aligned(conv_state, 16) ||
      !aligned(ssm, 16))
    return FL_ERR_INVALID_ARGUMENT;
  if (!workspace || workspace_bytes < mamba_step_bytes(B, heads)) return FL_ERR_WORKSPACE;
  if (!aligned(workspace, 16)) return FL_ERR_INVALID_ARGUMENT;
  const ConvParams conv{conv_w, conv_b, conv_dtype == FL_DTYPE_BF16};
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  const int nw16 = norm_dtype == FL_DTYPE_BF16, o16 = out_dtype == FL_DTYPE_BF16;
  return dtype == FL_DTYPE_BF16
             ? step_impl(static_cast<const bf16_bits*>(zxbcdt), B, heads, stride_b, conv, A_log, dt_bias, D, norm_w,
                         nw16, eps, conv_state, ssm, out, o16, ws, s)
             : step_impl(static_cast<const float*>(zxbcdt), B, heads, stride_b, conv, A_log, dt_bias, D, norm_w,
                         nw16, eps, conv_state, ssm, out, o16, ws, s);
}

}  // extern "C"
