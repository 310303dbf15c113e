// exact.hip — elementwise work of the refresh and Mamba-2 blocks in the stock ops' own roundings, bit
// for bit, so that it may run under autocast too, where a generation loop keeps its bits (reference:
// src/fields_official/reference/official_source/field_fusion_system_smoke_v21.py:131-253,
// field_fusion_wiki100_mamba2_v25.py:73-91). bf16 values are
// rounded after every operation, as an op on bf16 tensors does; sums and products with an order of
// their own (the matrix products, softmax) stay with the stock ops.
//
// Built with -ffp-contract=on: products and sums of separate statements stay separate.
#include "fl_common.h"

#pragma clang fp contract(off)

namespace {

using namespace fl;

constexpr int kHd = 64;

__device__ __forceinline__ float bf(const bf16_bits* p) { return load_as<bf16_bits>(p); }

// (a, b) -> (a cos - b sin, b cos + a sin), each product and each sum rounded
__device__ __forceinline__ void rope_pair(float a, float b, float c, float s, bf16_bits* first, bf16_bits* second) {
  const float ac = bf16_round(a * c), bs = bf16_round(b * s), bc = bf16_round(b * c), as = bf16_round(a * s);
  *first = (bf16_bits)bf16_bits_of(ac - bs);
  *second = (bf16_bits)bf16_bits_of(bc + as);
}

struct StepArgs {
  const bf16_bits* qlat;  // [B, q_heads * 64 + latent]
  const bf16_bits* kv;    // [B, 2 * kv_heads * 64]
  const bf16_bits* cos;   // [rope_len, 32]
  const bf16_bits* sin;
  const int64_t* pos;
  int q_heads, kv_heads, latent, rope_len, window, chunk, slots;
};

// One token's rotations and state writes before the attention: some 40 stock launches of 4 us in one.
// q [B, q_heads * 64] rotated; keys and values into the window's slot; the chunk's running latent sum
// (restarted on a chunk's first token) and its mean.
__global__ __launch_bounds__(256) void fl_refresh_step_in_kernel(StepArgs a, bf16_bits* __restrict__ q,
                                                                 bf16_bits* __restrict__ kt,
                                                                 bf16_bits* __restrict__ v,
                                                                 float* __restrict__ lat_sum,
                                                                 bf16_bits* __restrict__ mean) {
  const int64_t b = blockIdx.x, p = *a.pos;
  const int64_t at = p < a.rope_len - 1 ? (p < 0 ? 0 : p) : a.rope_len - 1;
  const int slot = (int)(((p % a.window) + a.window) % a.window);
  const bf16_bits *c = a.cos + at * 32, *s = a.sin + at * 32;
  const int qw = a.q_heads * kHd;
  const bf16_bits* x = a.qlat + b * (qw + a.latent);
  const bf16_bits* kv = a.kv + b * 2 * a.kv_heads * kHd;
  for (int i = threadIdx.x; i < a.q_heads * 32; i += 256) {
    const int o = (i >> 5) * kHd + (i & 31);
    rope_pair(bf(x + o), bf(x + o + 32), bf(c + (i & 31)), bf(s + (i & 31)), q + b * qw + o, q + b * qw + o + 32);
  }
  for (int i = threadIdx.x; i < a.kv_heads * 32; i += 256) {
    const int h = i >> 5, d = i & 31;
    bf16_bits* k = kt + ((b * a.kv_heads + h) * kHd + d) * a.window + slot;
    rope_pair(bf(kv + h * kHd + d), bf(kv + h * kHd + d + 32), bf(c + d), bf(s + d), k, k + (int64_t)32 * a.window);
  }
  for (int i = threadIdx.x; i < a.kv_heads * kHd; i += 256)
    v[((b * a.kv_heads + (i >> 6)) * a.window + slot) * kHd + (i & 63)] = kv[a.kv_heads * kHd + i];
  const float keep = ((p % a.chunk) + a.chunk) % a.chunk == 0 ? 0.f : 1.f, inv = 1.0f / (float)a.chunk;
  for (int i = threadIdx.x; i < a.latent; i += 256) {
    float t = lat_sum[b * a.latent + i] * keep;
    t = t + bf(x + qw + i);
    lat_sum[b * a.latent + i] = t;
    mean[b * a.latent + i] = (bf16_bits)bf16_bits_of(t * inv);  // a power of two: exact
  }
}

// The chunk's landmark of one token's running mean into its slot (clamped into the buffer).
__global__ __launch_bounds__(256) void fl_refresh_step_out_kernel(StepArgs a, bf16_bits* __restrict__ lkt,
                                                                  bf16_bits* __restrict__ lv) {
  const int64_t b = blockIdx.x, p = *a.pos;
  const int64_t at = p < a.rope_len - 1 ? (p < 0 ? 0 : p) : a.rope_len - 1;
  const int64_t chunk = p < 0 ? -1 : p / a.chunk;
  const int slot = (int)(chunk + 1 < a.slots - 1 ? chunk + 1 : a.slots - 1);
  const bf16_bits *c = a.cos + at * 32, *s = a.sin + at * 32;
  const bf16_bits* kv = a.kv + b * 2 * a.kv_heads * kHd;
  for (int i = threadIdx.x; i < a.kv_heads * 32; i += 256) {
    const int h = i >> 5, d = i & 31;
    bf16_bits* k = lkt + ((b * a.kv_heads + h) * kHd + d) * a.slots + slot;
    rope_pair(bf(kv + h * kHd + d), bf(kv + h * kHd + d + 32), bf(c + d), bf(s + d), k, k + (int64_t)32 * a.slots);
  }
  for (int i = threadIdx.x; i < a.kv_heads * kHd; i += 256)
    lv[((b * a.kv_heads + (i >> 6)) * a.slots + slot) * kHd + (i & 63)] = kv[a.kv_heads * kHd + i];
}

// out = float(scores) * scale where column j is visible, else -inf. Visible: j <= limit, with limit the
// token's window slot or its chunk (read from pos, period and step), or the row's index within lq
// (causal), or any. Four passes of the stock ops over the fp32 scores in one, bound by memory; for rows past
// 1,024 columns, which fl_masked_softmax_kernel does not hold.
__global__ __launch_bounds__(256) void fl_mask_scores_kernel(const bf16_bits* __restrict__ scores, uint64_t n,
                                                             uint32_t lk, uint32_t lq, int mode,
                                                             const int64_t* __restrict__ pos, int period,
                                                             float scale, float* __restrict__ out) {
  const uint64_t i = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= n) return;
  const uint64_t row = i / lk;
  const uint32_t j = (uint32_t)(i - row * lk);  // lk is a multiple of 4: one row per thread
  int64_t limit = lk;
  if (mode == 0) limit = row % lq;
  else if (mode == 1) limit = ((*pos % period) + period) % period;
  else limit = *pos / period;
  const u32x2 w = *reinterpret_cast<const u32x2*>(scores + i);
  const float s[4] = {bf16_lo(w.x), bf16_hi(w.x), bf16_lo(w.y), bf16_hi(w.y)};
  f32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = (int64_t)j + e <= limit ? s[e] * scale : -INFINITY;
  *reinterpret_cast<f32x4*>(out + i) = o;
}

__global__ __launch_bounds__(256) void fl_mask_scores_any_kernel(const bf16_bits* __restrict__ scores, uint64_t n,
                                                                 uint32_t lk, uint32_t lq, int mode,
                                                                 const int64_t* __restrict__ pos, int period,
                                                                 float scale, float* __restrict__ out) {
  const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint64_t row = i / lk;
  const int64_t j = (int64_t)(i - row * lk);
  const int64_t limit = mode == 0 ? (int64_t)(row % lq)
                                  : mode == 1 ? ((*pos % period) + period) % period : *pos / period;
  out[i] = j <= limit ? bf(scores + i) * scale : -INFINITY;
}

// v / sum as the division rounds it, from r = 1 / sum: the first residual brings the quotient within an
// ulp, the second rounds it correctly (Markstein, IBM J. Res. Dev. 34, 1990) as long as the residual is
// exact, which v >= 2^-80 keeps far from underflow; zeros stay zeros.
__device__ __forceinline__ float quotient(float v, float sum, float r) {
  float q = v * r;
  q = __builtin_fmaf(__builtin_fmaf(-q, sum, v), r, q);
  q = __builtin_fmaf(__builtin_fmaf(-q, sum, v), r, q);
  if (__any(v < 0x1p-80f && v > 0.f)) q = v / sum;
  return q;
}

// p = bf16(softmax(float(scores) * scale over the visible columns)), lk <= W IT columns, 64 / W rows per
// wave. The sum is the stock softmax's own up to 1,024 columns: lane l adds columns l, l + 64, ... in turn,
// then the lanes fold in halves, 32 down to 1; hidden columns add zeros, so they are neither read nor
// computed, and a row of at most W < 64 folds from W / 2. One pass of 4 bytes a score where mask, softmax
// and conversion moved 20: 134 M causal scores in rows of 1,024 took 400 us in three kernels and take 180
// (215 with a division per element); bound by the exponentials, quotients and 2-byte stores.
template <int IT, int W>
__global__ __launch_bounds__(256) void fl_masked_softmax_kernel(const bf16_bits* __restrict__ scores, uint64_t rows,
                                                                int lk, uint32_t lq, int mode,
                                                                const int64_t* __restrict__ pos, int period,
                                                                float scale, bf16_bits* __restrict__ out) {
  const int lane = threadIdx.x & (W - 1);
  const uint32_t sub = W == 64 ? __builtin_amdgcn_readfirstlane(threadIdx.x / 64) : threadIdx.x / W;
  const uint64_t row = (uint64_t)blockIdx.x * (256 / W) + sub;
  if (row >= rows) return;
  int64_t limit;
  if (mode == 0) limit = (uint32_t)row % lq;
  else if (mode == 1) limit = ((*pos % period) + period) % period;
  else if (mode == 2) limit = *pos / period;
  else limit = (uint32_t)row % lq / (uint32_t)period;
  const int n = limit < lk - 1 ? (limit < 0 ? 0 : (int)limit + 1) : lk;  // visible columns
  const bf16_bits* x = scores + row * lk;
  bf16_bits* y = out + row * lk;
  float v[IT], top = -INFINITY, sum = 0.f;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    v[i] = -INFINITY;
    if (W * i < n && lane + W * i < n) v[i] = bf(x + lane + W * i) * scale;
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) top = fmaxf(top, v[i]);
#pragma unroll
  for (int d = W / 2; d > 0; d >>= 1) top = fmaxf(top, __shfl_xor(top, d));
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    if (W * i < n) {
      v[i] = lane + W * i < n ? expf(v[i] - top) : 0.f;
      sum += v[i];
    }
  }
#pragma unroll
  for (int d = W / 2; d > 0; d >>= 1) sum += __shfl_xor(sum, d);
  const float r = 1.0f / sum, hidden = 0.f * r;  // NaN where the row's sum is NaN, or 0 (nothing visible)
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const float q = W * i < n ? quotient(v[i], sum, r) : hidden;
    if (lane + W * i < lk) y[lane + W * i] = (bf16_bits)bf16_bits_of(q);
  }
}

// out = y + round(sigmoid(mix)) * g, rounded after each operation
__global__ __launch_bounds__(256) void fl_mix_kernel(const bf16_bits* __restrict__ y, const bf16_bits* __restrict__ g,
                                                     const void* mix, int mix16, uint32_t n,
                                                     bf16_bits* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const float x = mix16 ? bf(static_cast<const bf16_bits*>(mix)) : *static_cast<const float*>(mix);
  const float s = bf16_round(1.0f / (1.0f + expf(-x)));
  const float t = bf16_round(s * bf(g + i));
  out[i] = (bf16_bits)bf16_bits_of(bf(y + i) + t);
}

// out = x + round(sigmoid(gate)) * a, rounded after each operation: three passes of the stock ops in one,
// bound by memory in a prompt and by the launch in a step. A multiple of 8 values, 16 bytes each.
__global__ __launch_bounds__(256) void fl_gate_add_kernel(const bf16_bits* __restrict__ x,
                                                          const bf16_bits* __restrict__ gate,
                                                          const bf16_bits* __restrict__ a, uint32_t n8,
                                                          bf16_bits* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n8) return;
  const int64_t at = (int64_t)i * 8;
  float v[8], g[8], w[8];
  Vec<bf16_bits, 8>::load(x + at, v);
  Vec<bf16_bits, 8>::load(gate + at, g);
  Vec<bf16_bits, 8>::load(a + at, w);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float s = bf16_round(1.0f / (1.0f + expf(-g[e])));
    v[e] += bf16_round(s * w[e]);
  }
  Vec<bf16_bits, 8>::store(out + at, v);
}

// ---- a prompt's heads ----

// 8 values from element o of each half of a head, rotated (8 pairs); zeros past the prompt
struct Rotated {
  bf16_bits first[8], second[8];
};
__device__ __forceinline__ Rotated rotate8(const bf16_bits* x, const bf16_bits* cos, const bf16_bits* sin) {
  float a[8], b[8], c[8], s[8];
  Vec<bf16_bits, 8>::load(x, a);
  Vec<bf16_bits, 8>::load(x + 32, b);
  Vec<bf16_bits, 8>::load(cos, c);
  Vec<bf16_bits, 8>::load(sin, s);
  Rotated r;
#pragma unroll
  for (int e = 0; e < 8; ++e) rope_pair(a[e], b[e], c[e], s[e], &r.first[e], &r.second[e]);
  return r;
}
__device__ __forceinline__ void put8(bf16_bits* p, const bf16_bits* v) {
  u32x4 w;
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = (uint32_t)v[2 * e] | (uint32_t)v[2 * e + 1] << 16;
  *reinterpret_cast<u32x4*>(p) = w;
}

// Queries of a prompt, rotated, in both orders the products read: q [B, heads, T, 64] and, zero-padded to
// whole windows of w, local [B, windows, heads, w, 64]. Four products, two sums, a concatenation and two
// copies of the stock ops (17 MB each way at 8,192 tokens of 16 heads) in one pass, bound by memory; with the
// two kernels below 230 us less per block of a 4 x 2,048 prompt.
__global__ __launch_bounds__(256) void fl_rope_queries_kernel(const bf16_bits* __restrict__ x, int64_t sb, int64_t st,
                                                              const bf16_bits* __restrict__ cos,
                                                              const bf16_bits* __restrict__ sin, uint32_t n, int T,
                                                              int heads, int w, int windows,
                                                              bf16_bits* __restrict__ q,
                                                              bf16_bits* __restrict__ local) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int o = (i & 3) * 8;
  const uint32_t r = i >> 2, h = r % (uint32_t)heads, row = r / (uint32_t)heads;
  const uint32_t padded = (uint32_t)(w * windows), t = row % padded, b = row / padded;
  Rotated v = {};
  if (t < (uint32_t)T) {
    v = rotate8(x + (int64_t)b * sb + (int64_t)t * st + h * kHd + o, cos + (int64_t)t * 32 + o, sin + (int64_t)t * 32 + o);
    bf16_bits* p = q + (((int64_t)b * heads + h) * T + t) * kHd + o;
    put8(p, v.first);
    put8(p + 32, v.second);
  }
  bf16_bits* p = local + ((((int64_t)b * windows + t / (uint32_t)w) * heads + h) * w + t % (uint32_t)w) * kHd + o;
  put8(p, v.first);
  put8(p + 32, v.second);
}

// Keys, rotated and transposed, kt [B, windows, heads, 64, w], and values v [B, windows, heads, w, 64] of a
// prompt, zero-padded: a lane holds a token, so that its wave's 2-byte stores of one dimension are adjacent.
__global__ __launch_bounds__(256) void fl_rope_keys_kernel(const bf16_bits* __restrict__ kv, int64_t sb, int64_t st,
                                                           const bf16_bits* __restrict__ cos,
                                                           const bf16_bits* __restrict__ sin, int T, int heads, int w,
                                                           int windows, bf16_bits* __restrict__ kt,
                                                           bf16_bits* __restrict__ v) {
  const int t = blockIdx.x * 64 + (threadIdx.x & 63), part = threadIdx.x >> 6, h = blockIdx.y;
  const int64_t b = blockIdx.z;
  if (t >= w * windows) return;
  Rotated k = {};
  u32x4 lo = {}, hi = {};
  if (t < T) {
    const bf16_bits* x = kv + b * sb + (int64_t)t * st + h * kHd;
    k = rotate8(x + part * 8, cos + (int64_t)t * 32 + part * 8, sin + (int64_t)t * 32 + part * 8);
    const u32x4* p = reinterpret_cast<const u32x4*>(x + heads * kHd + part * 16);
    lo = p[0];
    hi = p[1];
  }
  const int64_t base = ((b * windows + t / w) * heads + h) * (int64_t)w * kHd;
  bf16_bits* p = kt + base + t % w;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    p[(int64_t)(part * 8 + e) * w] = k.first[e];
    p[(int64_t)(part * 8 + 32 + e) * w] = k.second[e];
  }
  u32x4* y = reinterpret_cast<u32x4*>(v + base + (int64_t)(t % w) * kHd + part * 16);
  y[0] = lo;
  y[1] = hi;
}

// out [B, T, heads * 64] = local + round(sigmoid(mix)) * g, local in windows as above, g [B, heads, T, 64] or
// null for zeros; rounded after each operation
__global__ __launch_bounds__(256) void fl_mix_heads_kernel(const bf16_bits* __restrict__ local,
                                                           const bf16_bits* __restrict__ g, const void* mix, int mix16,
                                                           uint32_t n, int T, int heads, int w, int windows,
                                                           bf16_bits* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t r = i >> 3, h = r % (uint32_t)heads, row = r / (uint32_t)heads;
  const uint32_t t = row % (uint32_t)T, b = row / (uint32_t)T;
  const int o = (i & 7) * 8;
  const float x = mix16 ? bf(static_cast<const bf16_bits*>(mix)) : *static_cast<const float*>(mix);
  const float s = bf16_round(1.0f / (1.0f + expf(-x)));
  float a[8], c[8] = {};
  Vec<bf16_bits, 8>::load(
      local + ((((int64_t)b * windows + t / (uint32_t)w) * heads + h) * w + t % (uint32_t)w) * kHd + o, a);
  if (g) Vec<bf16_bits, 8>::load(g + (((int64_t)b * heads + h) * T + t) * kHd + o, c);
#pragma unroll
  for (int e = 0; e < 8; ++e) a[e] += bf16_round(s * c[e]);
  Vec<bf16_bits, 8>::store(out + (int64_t)i * 8, a);
}

// ---- Mamba-2 ----

// silu(bias + sum_k w[k] in[t - 3 + k]) of bf16 rows in fp32, each product and each sum rounded, in the
// stock order: a chain of five fp32 passes (75 MB each at 8,192 tokens) in one.
__global__ __launch_bounds__(256) void fl_conv_silu_kernel(const bf16_bits* __restrict__ x, int64_t sb, int64_t st,
                                                           int L, int channels, const void* w, const void* bias,
                                                           int is16, float* __restrict__ out) {
  const int c = blockIdx.x * 256 + threadIdx.x, t0 = blockIdx.y * 16;
  const int64_t b = blockIdx.z;
  if (c >= channels) return;
  float wt[4], bs;
  if (is16) {
    for (int k = 0; k < 4; ++k) wt[k] = bf(static_cast<const bf16_bits*>(w) + 4 * c + k);
    bs = bf(static_cast<const bf16_bits*>(bias) + c);
  } else {
    for (int k = 0; k < 4; ++k) wt[k] = static_cast<const float*>(w)[4 * c + k];
    bs = static_cast<const float*>(bias)[c];
  }
  const bf16_bits* p = x + b * sb + c;
  float in[19];
#pragma unroll
  for (int i = 0; i < 19; ++i) {
    const int t = t0 - 3 + i;
    in[i] = bf(p + (int64_t)min(max(t, 0), L - 1) * st);
    if (t < 0) in[i] = 0.f;
  }
  float* o = out + (b * L + t0) * channels + c;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    if (t0 + i >= L) break;
    float v = in[i] * wt[0];
    v = bs + v;
#pragma unroll
    for (int k = 1; k < 4; ++k) {
      const float m = in[i + k] * wt[k];
      v = v + m;
    }
    o[(int64_t)i * channels] = v / (1.0f + expf(-v));
  }
}

// [b, h, c, s, s] = cb[b, c] * exp(acs_i - acs_j) for j <= i, times 0 above, rounded to the bf16 operand
// that autocast makes of it: six fp32 passes over the largest tensor of the block in one, bound by its
// writes. 134 MB of weights (4 x 2,048 tokens, 32 heads) take 47 us, 2.9 TB/s; 126 us with a branch and a
// 4-byte load of acs per element.
__global__ __launch_bounds__(256) void fl_decay_product_kernel(const bf16_bits* __restrict__ cb,
                                                               const float* __restrict__ acs, int H, int n_chunks,
                                                               int s, bf16_bits* __restrict__ out) {
  const int row_vecs = s / 8;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= s * row_vecs) return;
  const int i = idx / row_vecs, j0 = 8 * (idx - i * row_vecs), c = blockIdx.y;
  const int64_t bh = blockIdx.z, b = bh / H;
  const float* a = acs + (bh * n_chunks + c) * s;
  float v[8], o[8], aj[8];
  Vec<bf16_bits, 8>::load(cb + ((b * n_chunks + c) * s + i) * s + j0, v);
  if (j0 <= i) {
    Vec<float, 8>::load(a + j0, aj);
    const float ai = a[i];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = expf(ai - aj[e]);  // beside the diagonal too: a select costs less than eight branches
      o[e] = v[e] * (j0 + e <= i ? d : 0.f);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = v[e] * 0.f;
  }
  Vec<bf16_bits, 8>::store(out + (((bh * n_chunks + c) * s + i) * s + j0), o);
}

// The two operands autocast makes of x dt, each bf16 of fp32 products: xdt [B, H, chunks, s, P] and, times
// w_end (the decay to the chunk's end), xw [B, H, chunks, P, s], zeros past L. A tile of 64 tokens by 64
// dimensions goes through LDS, so that both orders are read and written in rows. Two products, two
// reorderings and two conversions of the stock ops in fp32 (67 MB each way at 8,192 tokens) in one pass.
__global__ __launch_bounds__(256) void fl_ssd_operands_kernel(const float* __restrict__ x, int64_t sb, int64_t st,
                                                              const float* __restrict__ dt, int64_t dt_sb,
                                                              const float* __restrict__ w_end, int H, int n_chunks,
                                                              int s, int P, int64_t L, bf16_bits* __restrict__ xdt,
                                                              bf16_bits* __restrict__ xw) {
  __shared__ bf16_bits tile[64][66];
  const int s_tiles = (s + 63) / 64, t0 = (int)(blockIdx.x % s_tiles) * 64, p0 = (int)(blockIdx.x / s_tiles) * 64;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, h = (int)(blockIdx.z % H);
  const int64_t b = blockIdx.z / H, bhc = (int64_t)blockIdx.z * n_chunks + blockIdx.y;
  const int64_t first = (int64_t)blockIdx.y * s + t0;  // the tile's first token
  const bool has = p0 + lane < P;
  for (int t = wave; t < 64 && t0 + t < s; t += 4) {
    float v = 0.f;
    if (has && first + t < L)
      v = x[b * sb + (first + t) * st + (int64_t)h * P + p0 + lane] * dt[b * dt_sb + (first + t) * H + h];
    if (has) xdt[(bhc * s + t0 + t) * P + p0 + lane] = (bf16_bits)bf16_bits_of(v);
    const float w = v * w_end[bhc * s + t0 + t];
    tile[lane][t] = (bf16_bits)bf16_bits_of(w);
  }
  __syncthreads();
  if (t0 + lane < s)
    for (int d = wave; d < 64 && p0 + d < P; d += 4) xw[(bhc * P + p0 + d) * s + t0 + lane] = tile[d][lane];
}

// What the gated norm takes the mean square of: ((y + y_off exp(acs)) + D x) silu(z), each operation rounded
// in fp32, [B, L, H P] from y and y_off [B, H, chunks, s, P]: eight fp32 passes in one, bound by memory.
__global__ __launch_bounds__(256) void fl_ssd_finish_kernel(const bf16_bits* __restrict__ y,
                                                            const bf16_bits* __restrict__ y_off,
                                                            const float* __restrict__ acs,
                                                            const float* __restrict__ x, int64_t x_sb, int64_t x_st,
                                                            const float* __restrict__ D,
                                                            const bf16_bits* __restrict__ z, int64_t z_sb, int64_t z_st,
                                                            uint32_t n, int H, int n_chunks, int s, int P, int L,
                                                            float* __restrict__ out) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t width = (uint32_t)(H * P / 4), row = i / width, col = (i - row * width) * 4;
  const uint32_t b = row / (uint32_t)L, t = row - b * (uint32_t)L, h = col / (uint32_t)P, p = col - h * (uint32_t)P;
  const uint32_t c = t / (uint32_t)s;
  const int64_t at = (((int64_t)b * H + h) * n_chunks + c) * s + (t - c * (uint32_t)s);
  auto load4 = [](const bf16_bits* q, float* o) {
    const u32x2 w = *reinterpret_cast<const u32x2*>(q);
    o[0] = bf16_lo(w.x), o[1] = bf16_hi(w.x), o[2] = bf16_lo(w.y), o[3] = bf16_hi(w.y);
  };
  float a[4], off[4], g[4];
  load4(y + at * P + p, a);
  load4(y_off + at * P + p, off);
  load4(z + (int64_t)b * z_sb + (int64_t)t * z_st + col, g);
  const f32x4 xv = *reinterpret_cast<const f32x4*>(x + (int64_t)b * x_sb + (int64_t)t * x_st + col);
  const float e = expf(acs[at]), d = D[h];
  f32x4 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float m = off[k] * e, u = a[k] + m, dx = d * xv[k], v = u + dx;
    const float silu = g[k] / (1.0f + expf(-g[k]));
    o[k] = v * silu;
  }
  *reinterpret_cast<f32x4*>(out + (int64_t)i * 4) = o;
}

// One token's state update, s = s * decay then s + xdt * b, each rounded, and the bf16 operand that
// autocast makes of the state for its product with C: 500 MB of traffic in 168 MB at 64 x 32 heads.
__global__ __launch_bounds__(256) void fl_state_update_kernel(const float* __restrict__ decay,
                                                              const float* __restrict__ xdt,
                                                              const float* __restrict__ bm, int64_t bm_stride,
                                                              int H, int P, int N, float* __restrict__ ssm,
                                                              bf16_bits* __restrict__ ssm16) {
  const int64_t bh = blockIdx.x, b = bh / H;
  const float d = decay[bh];
  for (int i = threadIdx.x; i < P * N / 4; i += 256) {
    const int p = 4 * i / N, n = 4 * i - p * N;
    float* at = ssm + bh * P * N + 4 * (int64_t)i;
    f32x4 v = *reinterpret_cast<const f32x4*>(at);
    const float x = xdt[bh * P + p];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float t = x * bm[b * bm_stride + n + e];
      const float q = v[e] * d;
      v[e] = q + t;
    }
    *reinterpret_cast<f32x4*>(at) = v;
    u32x2 w;
    w.x = bf16_pair(v[0], v[1]);
    w.y = bf16_pair(v[2], v[3]);
    *reinterpret_cast<u32x2*>(ssm16 + bh * P * N + 4 * (int64_t)i) = w;
  }
}

bool step_ok(const StepArgs& a, int64_t B) {
  return B > 0 && B <= (1 << 20) && a.q_heads > 0 && a.q_heads <= 4096 && a.kv_heads > 0 && a.kv_heads <= 4096 &&
         a.latent > 0 && a.latent <= (1 << 16) && a.rope_len > 0 && a.window > 0 && a.chunk > 0 &&
         (a.chunk & (a.chunk - 1)) == 0 && a.slots > 0 && a.kv && a.cos && a.sin && a.pos;
}

StepArgs step_args(const void* qlat, const void* kv, const void* cos, const void* sin, const int64_t* pos,
                   int64_t q_heads, int64_t kv_heads, int64_t latent, int64_t rope_len, int64_t window, int64_t chunk,
                   int64_t slots) {
  auto p = [](const void* t) { return static_cast<const bf16_bits*>(t); };
  return {p(qlat), p(kv), p(cos), p(sin), pos, (int)q_heads, (int)kv_heads, (int)latent, (int)rope_len,
          (int)window, (int)chunk, (int)slots};
}

}  // namespace

extern "C" {

int fl_refresh_step_in(const void* qlat, const void* kv, const void* cos, const void* sin, const int64_t* pos,
                       int64_t B, int64_t q_heads, int64_t kv_heads, int64_t latent, int64_t rope_len, int64_t window,
                       int64_t chunk, void* q, void* kt, void* v, float* lat_sum, void* mean, void* stream) {
  const StepArgs a = step_args(qlat, kv, cos, sin, pos, q_heads, kv_heads, latent, rope_len, window, chunk, 1);
  if (rope_len > (1 << 28) || window > (1 << 28) || chunk > (1 << 28) || !step_ok(a, B) || !qlat || !q || !kt || !v ||
      !lat_sum || !mean)
    return FL_ERR_INVALID_ARGUMENT;
  fl_refresh_step_in_kernel<<<(unsigned)B, 256, 0, static_cast<hipStream_t>(stream)>>>(
      a, static_cast<bf16_bits*>(q), static_cast<bf16_bits*>(kt), static_cast<bf16_bits*>(v), lat_sum,
      static_cast<bf16_bits*>(mean));
  return hip_status(hipGetLastError());
}

int fl_refresh_step_out(const void* kv, const void* cos, const void* sin, const int64_t* pos, int64_t B,
                        int64_t kv_heads, int64_t rope_len, int64_t chunk, int64_t slots, void* lkt, void* lv,
                        void* stream) {
  const StepArgs a = step_args(nullptr, kv, cos, sin, pos, 1, kv_heads, 1, rope_len, 1, chunk, slots);
  if (rope_len > (1 << 28) || chunk > (1 << 28) || slots > (1 << 28) || !step_ok(a, B) || !lkt || !lv)
    return FL_ERR_INVALID_ARGUMENT;
  fl_refresh_step_out_kernel<<<(unsigned)B, 256, 0, static_cast<hipStream_t>(stream)>>>(
      a, static_cast<bf16_bits*>(lkt), static_cast<bf16_bits*>(lv));
  return hip_status(hipGetLastError());
}

int fl_mask_scores(const void* scores, int64_t rows, int64_t lk, int64_t lq, int mode, const int64_t* pos,
                   int64_t period, float scale, float* out, void* stream) {
  if (rows <= 0 || lk <= 0 || lq <= 0 || rows > ((int64_t)1 << 40) / lk || lk > (1 << 30) || lq > (1 << 30) ||
      mode < 0 || mode > 2 || (mode > 0 && (!pos || period <= 0 || period > (1 << 30))) || !scores || !out)
    return FL_ERR_INVALID_ARGUMENT;
  const int64_t n = rows * lk;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bf16_bits* p = static_cast<const bf16_bits*>(scores);
  const bool vec = lk % 4 == 0 && aligned(scores, 8) && aligned(out, 16);
  if (cdiv(n, vec ? 1024 : 256) >= ((int64_t)1 << 31)) return FL_ERR_INVALID_ARGUMENT;
  if (vec) {
    fl_mask_scores_kernel<<<(unsigned)cdiv(n, 1024), 256, 0, s>>>(p, (uint64_t)n, (uint32_t)lk, (uint32_t)lq, mode, pos,
                                                                  (int)period, scale, out);
  } else {
    fl_mask_scores_any_kernel<<<(unsigned)cdiv(n, 256), 256, 0, s>>>(p, (uint64_t)n, (uint32_t)lk, (uint32_t)lq, mode,
                                                                     pos, (int)period, scale, out);
  }
  return hip_status(hipGetLastError());
}

int fl_masked_softmax(const void* scores, int64_t rows, int64_t lk, int64_t lq, int mode, const int64_t* pos,
                      int64_t period, float scale, void* out, void* stream) {
  if (rows <= 0 || rows > ((int64_t)1 << 32) - 1 || lk <= 0 || lk > 1024 || lq <= 0 || lq > (1 << 30) || mode < 0 ||
      mode > 3 || ((mode == 1 || mode == 2) && !pos) || (mode > 0 && (period <= 0 || period > (1 << 30))) || !scores ||
      !out)
    return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bf16_bits* x = static_cast<const bf16_bits*>(scores);
  auto run = [&](auto kernel, int per_block) {
    kernel<<<(unsigned)cdiv(rows, per_block), 256, 0, s>>>(x, (uint64_t)rows, (int)lk, (uint32_t)lq, mode, pos,
                                                           (int)period, scale, static_cast<bf16_bits*>(out));
  };
  // the fewest lanes, then the fewest columns per lane, that hold a row
  if (lk <= 16) run(fl_masked_softmax_kernel<1, 16>, 16);
  else if (lk <= 32) run(fl_masked_softmax_kernel<1, 32>, 8);
  else if (lk <= 64) run(fl_masked_softmax_kernel<1, 64>, 4);
  else if (lk <= 128) run(fl_masked_softmax_kernel<2, 64>, 4);
  else if (lk <= 256) run(fl_masked_softmax_kernel<4, 64>, 4);
  else if (lk <= 512) run(fl_masked_softmax_kernel<8, 64>, 4);
  else run(fl_masked_softmax_kernel<16, 64>, 4);
  return hip_status(hipGetLastError());
}

int fl_rope_heads(const void* x, int64_t x_stride_b, int64_t x_stride_t, const void* kv, int64_t kv_stride_b,
                  int64_t kv_stride_t, const void* cos, const void* sin, int64_t B, int64_t T, int64_t q_heads,
                  int64_t kv_heads, int64_t window, void* q, void* local, void* kt, void* v, void* stream) {
  if (B <= 0 || B > 65535 || T <= 0 || T > (1 << 26) || window <= 0 || window > T || q_heads <= 0 || q_heads > 4096 ||
      kv_heads <= 0 || kv_heads > 4096 || x_stride_t < q_heads * kHd || kv_stride_t < 2 * kv_heads * kHd ||
      x_stride_b < 0 || kv_stride_b < 0 || (x_stride_b | x_stride_t | kv_stride_b | kv_stride_t) % 8 || !x || !kv ||
      !cos || !sin || !q || !local || !kt || !v)
    return FL_ERR_INVALID_ARGUMENT;
  for (const void* p : {x, kv, cos, sin, (const void*)q, (const void*)local, (const void*)v})
    if (!aligned(p, 16)) return FL_ERR_INVALID_ARGUMENT;
  const int64_t windows = cdiv(T, window), n = B * windows * window * q_heads * 4;
  if (n >= ((int64_t)1 << 31)) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto in = [](const void* p) { return static_cast<const bf16_bits*>(p); };
  auto to = [](void* p) { return static_cast<bf16_bits*>(p); };
  fl_rope_queries_kernel<<<(unsigned)cdiv(n, 256), 256, 0, s>>>(in(x), x_stride_b, x_stride_t, in(cos), in(sin),
                                                                (uint32_t)n, (int)T, (int)q_heads, (int)window,
                                                                (int)windows, to(q), to(local));
  fl_rope_keys_kernel<<<dim3((unsigned)cdiv(windows * window, 64), (unsigned)kv_heads, (unsigned)B), 256, 0, s>>>(
      in(kv), kv_stride_b, kv_stride_t, in(cos), in(sin), (int)T, (int)kv_heads, (int)window, (int)windows, to(kt),
      to(v));
  return hip_status(hipGetLastError());
}

int fl_mix_heads(const void* local, const void* g, const void* mix_logit, int mix_dtype, int64_t B, int64_t T,
                 int64_t heads, int64_t window, void* out, void* stream) {
  if (!dtype_ok(mix_dtype)) return FL_ERR_DTYPE;
  if (B <= 0 || T <= 0 || T > (1 << 26) || heads <= 0 || heads > 4096 || window <= 0 || window > T ||
      B > (((int64_t)1 << 31) - 1) / 8 / heads / T || !local || !mix_logit || !out || !aligned(local, 16) ||
      !aligned(out, 16) || (g && !aligned(g, 16)))
    return FL_ERR_INVALID_ARGUMENT;
  const int64_t n = B * T * heads * 8;
  fl_mix_heads_kernel<<<(unsigned)cdiv(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const bf16_bits*>(local), static_cast<const bf16_bits*>(g), mix_logit, mix_dtype == FL_DTYPE_BF16,
      (uint32_t)n, (int)T, (int)heads, (int)window, (int)cdiv(T, window), static_cast<bf16_bits*>(out));
  return hip_status(hipGetLastError());
}

int fl_gate_add(const void* x, const void* gate, const void* a, int64_t n, void* out, void* stream) {
  if (n <= 0 || n % 8 || n / 8 > ((int64_t)1 << 32) - 256 || !x || !gate || !a || !out || !aligned(x, 16) ||
      !aligned(gate, 16) || !aligned(a, 16) || !aligned(out, 16))
    return FL_ERR_INVALID_ARGUMENT;
  fl_gate_add_kernel<<<(unsigned)cdiv(n / 8, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const bf16_bits*>(x), static_cast<const bf16_bits*>(gate), static_cast<const bf16_bits*>(a),
      (uint32_t)(n / 8), static_cast<bf16_bits*>(out));
  return hip_status(hipGetLastError());
}

int fl_conv_silu(const void* x, int64_t stride_b, int64_t stride_t, int64_t B, int64_t L, int64_t channels,
                 const void* w, const void* bias, int w_dtype, float* out, void* stream) {
  if (!dtype_ok(w_dtype)) return FL_ERR_DTYPE;
  if (B <= 0 || B > 65535 || L <= 0 || L > 65535 * 16 || channels <= 0 || channels > (1 << 24) ||
      stride_t < channels || stride_b < 0 || !x || !w || !bias || !out)
    return FL_ERR_INVALID_ARGUMENT;
  fl_conv_silu_kernel<<<dim3((unsigned)cdiv(channels, 256), (unsigned)cdiv(L, 16), (unsigned)B), 256, 0,
                        static_cast<hipStream_t>(stream)>>>(static_cast<const bf16_bits*>(x), stride_b, stride_t, (int)L,
                                                            (int)channels, w, bias, w_dtype == FL_DTYPE_BF16, out);
  return hip_status(hipGetLastError());
}

int fl_decay_product(const void* cb, const float* acs, int64_t B, int64_t heads, int64_t n_chunks, int64_t s,
                     void* out, void* stream) {
  if (B <= 0 || heads <= 0 || B * heads > 65535 || n_chunks <= 0 || n_chunks > 65535 || s <= 0 || s % 8 || s > 4096 ||
      !cb || !acs || !out || !aligned(cb, 16) || !aligned(acs, 16) || !aligned(out, 16))
    return FL_ERR_INVALID_ARGUMENT;
  fl_decay_product_kernel<<<dim3((unsigned)cdiv(s * (s / 8), 256), (unsigned)n_chunks, (unsigned)(B * heads)), 256, 0,
                            static_cast<hipStream_t>(stream)>>>(static_cast<const bf16_bits*>(cb), acs, (int)heads,
                                                                (int)n_chunks, (int)s, static_cast<bf16_bits*>(out));
  return hip_status(hipGetLastError());
}

int fl_ssd_operands(const float* x, int64_t x_stride_b, int64_t x_stride_t, const float* dt, int64_t dt_stride_b,
                    const float* w_end, int64_t B, int64_t heads, int64_t n_chunks, int64_t s, int64_t P, int64_t L,
                    void* xdt, void* xw, void* stream) {
  if (B <= 0 || heads <= 0 || B * heads > 65535 || n_chunks <= 0 || n_chunks > 65535 || s <= 0 || s > 4096 || P <= 0 ||
      P > 4096 || L <= 0 || L > n_chunks * s || x_stride_t < heads * P || x_stride_b < 0 || dt_stride_b < 0 || !x ||
      !dt || !w_end || !xdt || !xw)
    return FL_ERR_INVALID_ARGUMENT;
  fl_ssd_operands_kernel<<<dim3((unsigned)(cdiv(s, 64) * cdiv(P, 64)), (unsigned)n_chunks, (unsigned)(B * heads)), 256,
                           0, static_cast<hipStream_t>(stream)>>>(
      x, x_stride_b, x_stride_t, dt, dt_stride_b, w_end, (int)heads, (int)n_chunks, (int)s, (int)P, L,
      static_cast<bf16_bits*>(xdt), static_cast<bf16_bits*>(xw));
  return hip_status(hipGetLastError());
}

int fl_ssd_finish(const void* y, const void* y_off, const float* acs, const float* x, int64_t x_stride_b,
                  int64_t x_stride_t, const float* D, const void* z, int64_t z_stride_b, int64_t z_stride_t, int64_t B,
                  int64_t heads, int64_t n_chunks, int64_t s, int64_t P, int64_t L, float* out, void* stream) {
  if (B <= 0 || heads <= 0 || B * heads > 65535 || n_chunks <= 0 || n_chunks > 65535 || s <= 0 || s > 4096 || P <= 0 ||
      P > 4096 || P % 4 || L <= 0 || L > n_chunks * s || x_stride_t < heads * P || z_stride_t < heads * P ||
      x_stride_b < 0 || z_stride_b < 0 || (x_stride_b | x_stride_t | z_stride_b | z_stride_t) % 4 || !y || !y_off ||
      !acs || !x || !D || !z || !out || !aligned(y, 8) || !aligned(y_off, 8) || !aligned(x, 16) || !aligned(z, 8) ||
      !aligned(out, 16))
    return FL_ERR_INVALID_ARGUMENT;
  if (L > (((int64_t)1 << 32) - 256) / (heads * P / 4) / B) return FL_ERR_INVALID_ARGUMENT;
  const int64_t n = B * L * (heads * P / 4);
  fl_ssd_finish_kernel<<<(unsigned)cdiv(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const bf16_bits*>(y), static_cast<const bf16_bits*>(y_off), acs, x, x_stride_b, x_stride_t, D,
      static_cast<const bf16_bits*>(z), z_stride_b, z_stride_t, (uint32_t)n, (int)heads, (int)n_chunks, (int)s, (int)P,
      (int)L, out);
  return hip_status(hipGetLastError());
}

int fl_state_update(const float* decay, const float* xdt, const float* bm, int64_t bm_stride, int64_t B, int64_t heads,
                    int64_t P, int64_t N, float* ssm, void* ssm16, void* stream) {
  if (B <= 0 || heads <= 0 || B * heads > (1 << 30) || P <= 0 || N <= 0 || N % 4 || P * N > (1 << 24) ||
      bm_stride < N || !decay || !xdt || !bm || !ssm || !ssm16 || !aligned(ssm, 16) || !aligned(ssm16, 8))
    return FL_ERR_INVALID_ARGUMENT;
  fl_state_update_kernel<<<(unsigned)(B * heads), 256, 0, static_cast<hipStream_t>(stream)>>>(
      decay, xdt, bm, bm_stride, (int)heads, (int)P, (int)N, ssm, static_cast<bf16_bits*>(ssm16));
  return hip_status(hipGetLastError());
}

int fl_mix(const void* y, const void* g, const void* mix_logit, int mix_dtype, int64_t n, void* out, void* stream) {
  if (!dtype_ok(mix_dtype)) return FL_ERR_DTYPE;
  if (n <= 0 || n > ((int64_t)1 << 31) - 1 || !y || !g || !mix_logit || !out) return FL_ERR_INVALID_ARGUMENT;
  fl_mix_kernel<<<(unsigned)cdiv(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      static_cast<const bf16_bits*>(y), static_cast<const bf16_bits*>(g), mix_logit, mix_dtype == FL_DTYPE_BF16,
      (uint32_t)n, static_cast<bf16_bits*>(out));
  return hip_status(hipGetLastError());
}

}  // extern "C"
