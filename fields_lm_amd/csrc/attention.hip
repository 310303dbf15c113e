// attention.hip — the refresh blocks' attention over whole sequences (no gradient): RoPE, causal
// attention inside consecutive windows, causal attention to completed chunks' landmarks, and their
// mix (reference: src/fields_official/reference/official_source/field_fusion_system_smoke_v21.py:
// 131-253, RoPE field_fusion_300m_screen_v20.py:121-144). bf16 operands, head dimension 64, fp32
// scores, softmax and sums; and the plain RMSNorm of those blocks.
#include "fl_common.h"

namespace {

using namespace fl;

constexpr int kHd = 64;         // head dimension
constexpr int kQTile = 32;      // queries per wave
constexpr int kKTile = 64;      // keys per step
constexpr int kRow = kHd + 8;   // bf16 per staged row: 36 dwords, so that 16 rows' 16-byte reads take all banks

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 8 values rotated with their partners 32 dimensions on: (a, b) -> (a cos - b sin, b cos + a sin)
__device__ __forceinline__ void rotate(const bf16_bits* cos, const bf16_bits* sin, float* a, float* b) {
  float c[8], s[8];
  Vec<bf16_bits, 8>::load(cos, c);
  Vec<bf16_bits, 8>::load(sin, s);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = a[e], y = b[e];
    a[e] = fmaf(x, c[e], -(y * s[e]));
    b[e] = fmaf(y, c[e], x * s[e]);
  }
}

// ------------------------------------------------------------------------------------------
// Keys rotated, [B, heads, T, 64], and values transposed, [B, heads, 64, Tp] (Tp: T rounded up to
// 64, the rest zero), from kv rows [keys of all heads | values of all heads]: the attention reads its
// operands in the order the matrix instructions take them. Position of row t: pos0 + pos_step t.
// Bound by memory, 4 KB per token of 4 heads moved once.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fl_rope_kv_kernel(const bf16_bits* __restrict__ kv, int64_t sb,
                                                         int64_t st, int T, int Tp, int heads, int pos0,
                                                         int pos_step, const bf16_bits* __restrict__ cos,
                                                         const bf16_bits* __restrict__ sin,
                                                         bf16_bits* __restrict__ k_out,
                                                         bf16_bits* __restrict__ vt_out) {
  __shared__ bf16_bits s_v[64][kRow];
  const int h = blockIdx.y, b = blockIdx.z, t0 = blockIdx.x * 64;
  const int row = threadIdx.x >> 2, q8 = 8 * (threadIdx.x & 3), t = t0 + row;
  const bf16_bits* p = kv + b * sb + (int64_t)min(t, T - 1) * st + h * kHd;
  const bf16_bits* pv = p + heads * kHd;
  u32x4 v0 = *reinterpret_cast<const u32x4*>(pv + q8), v1 = *reinterpret_cast<const u32x4*>(pv + 32 + q8);
  if (t < T) {
    float a[8], c[8];
    Vec<bf16_bits, 8>::load(p + q8, a);
    Vec<bf16_bits, 8>::load(p + 32 + q8, c);
    const int64_t pos = pos0 + (int64_t)pos_step * t;
    rotate(cos + pos * 32 + q8, sin + pos * 32 + q8, a, c);
    bf16_bits* o = k_out + (((int64_t)b * heads + h) * T + t) * kHd;
    Vec<bf16_bits, 8>::store(o + q8, a);
    Vec<bf16_bits, 8>::store(o + 32 + q8, c);
  } else {
    v0 = v1 = u32x4{0u, 0u, 0u, 0u};
  }
  *reinterpret_cast<u32x4*>(&s_v[row][q8]) = v0;
  *reinterpret_cast<u32x4*>(&s_v[row][32 + q8]) = v1;
  __syncthreads();
  u32x4 o[2];  // dimension `row`, 16 tokens
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int c = 2 * q8 + 2 * e;
    o[e >> 2][e & 3] = (uint32_t)s_v[c][row] | (uint32_t)s_v[c + 1][row] << 16;
  }
  u32x4* dst = reinterpret_cast<u32x4*>(vt_out + (((int64_t)b * heads + h) * kHd + row) * Tp + t0 + 2 * q8);
  dst[0] = o[0];
  dst[1] = o[1];
}

// ------------------------------------------------------------------------------------------
// One block per (sequence, KV head, 32 queries): a wave per query head of the group, so that the
// group shares the staged keys and values. Scores are formed transposed (rows: keys), which leaves
// each lane one query's column: the softmax needs two cross-lane steps, and the probabilities are
// already the operand of the second product, with keys in the order (4 of one 16-key tile, 4 of the
// next) that the values are read in. Bound by the vector work of the softmax (some 12 operations per
// score against 4 cycles of products). 4 x 1,900 tokens, 16 / 4 heads, window 512: 38 us with the
// rotation of q and the landmarks (stock: some 1,050 us of scores, masks, softmax and copies).
// ------------------------------------------------------------------------------------------
struct Keys {
  const bf16_bits* k;   // [rows, 64]
  const bf16_bits* vt;  // [64, tp]
  int rows, tp;
};

template <int REP>
__global__ __launch_bounds__(64 * REP) void fl_window_attention_kernel(
    const bf16_bits* __restrict__ q, int64_t q_sb, int64_t q_st, int T, int Tp, int kv_heads, int window,
    const bf16_bits* __restrict__ k, const bf16_bits* __restrict__ vt, int n_land, int land_tp,
    int land_chunk, const bf16_bits* __restrict__ lk, const bf16_bits* __restrict__ lvt,
    const bf16_bits* __restrict__ cos, const bf16_bits* __restrict__ sin, const void* mix, int mix16,
    bf16_bits* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) bf16_bits s_k[kKTile][kRow], s_v[kHd][kRow];
  const int lane = threadIdx.x & 63, wave = uniform(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int t0 = blockIdx.x * kQTile, kvh = blockIdx.y, b = blockIdx.z, h = kvh * REP + wave;
  const int64_t kv_row = (int64_t)b * kv_heads + kvh;
  constexpr float kScale = 0.125f * kLog2e;  // 64^-1/2, base-2 exponents

  bf16x8 qf[2][2];  // [16-query tile][dimensions 0-31, 32-63]
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int t = min(t0 + 16 * tt + r, T - 1);
    const bf16_bits* p = q + b * q_sb + (int64_t)t * q_st + h * kHd + 8 * g;
    float a[8], c[8];
    Vec<bf16_bits, 8>::load(p, a);
    Vec<bf16_bits, 8>::load(p + 32, c);
    rotate(cos + (int64_t)t * 32 + 8 * g, sin + (int64_t)t * 32 + 8 * g, a, c);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      qf[tt][0][e] = (__bf16)a[e];
      qf[tt][1][e] = (__bf16)c[e];
    }
  }

  f32x4 o[4][2];  // [16-dimension tile][query tile]: dimensions 4 g + i of query r
  float m[2], l[2];
  constexpr int kPieces = 8 / REP;  // 16-byte pieces of a step's keys, and of its values, per thread
  u32x4 pk[kPieces], pv[kPieces];
  auto fetch = [&](const Keys& ks, int key0) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int id = threadIdx.x + i * 64 * REP, row = id >> 3, c = 8 * (id & 7);
      pk[i] = *reinterpret_cast<const u32x4*>(ks.k + (int64_t)min(key0 + row, ks.rows - 1) * kHd + c);
      pv[i] = *reinterpret_cast<const u32x4*>(ks.vt + (int64_t)row * ks.tp + key0 + c);
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const int id = threadIdx.x + i * 64 * REP, row = id >> 3, c = 8 * (id & 7);
      *reinterpret_cast<u32x4*>(&s_k[row][c]) = pk[i];
      *reinterpret_cast<u32x4*>(&s_v[row][c]) = pv[i];
    }
  };
  // attends to keys [first, end) of ks (end > first, first a multiple of 64); a query also stops at
  // last0 + its own index (its causal limit)
  auto attend = [&](const Keys& ks, int first, int end, int last0) {
    fetch(ks, first);
    for (int key0 = first; key0 < end; key0 += kKTile) {
      __syncthreads();  // every wave has read the previous step's tiles
      stage();
      __syncthreads();
      if (key0 + kKTile < end) fetch(ks, key0 + kKTile);
      f32x4 s[4][2];
#pragma unroll
      for (int kt = 0; kt < 4; ++kt) {
        s[kt][0] = s[kt][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const bf16x8 a = *reinterpret_cast<const bf16x8*>(&s_k[16 * kt + r][32 * d + 8 * g]);
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) s[kt][tt] = mfma32(a, qf[tt][d], s[kt][tt]);
        }
      }
      if (key0 + kKTile > min(end, last0 + 1)) {  // the step holds keys that some query must not see
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = key0 + 16 * kt + 4 * g + i;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
              if (key >= end || key > last0 + 16 * tt + r) s[kt][tt][i] = -INFINITY;
          }
      }
      bf16x8 p[2][2];  // [32-key half][query tile]
#pragma unroll
      for (int tt = 0; tt < 2; ++tt) {
        float mx = m[tt];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) mx = fmaxf(mx, s[kt][tt][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float alpha = __builtin_amdgcn_exp2f((m[tt] - mx) * kScale), off = -mx * kScale;
        m[tt] = mx;
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float e = __builtin_amdgcn_exp2f(fmaf(s[kt][tt][i], kScale, off));
            sum += e;
            p[kt >> 1][tt][4 * (kt & 1) + i] = (__bf16)e;
          }
        l[tt] = fmaf(l[tt], alpha, sum);
#pragma unroll
        for (int ht = 0; ht < 4; ++ht) o[ht][tt] *= alpha;
      }
#pragma unroll
      for (int ht = 0; ht < 4; ++ht)
#pragma unroll
        for (int kp = 0; kp < 2; ++kp) {
          const bf16x4 a0 = *reinterpret_cast<const bf16x4*>(&s_v[16 * ht + r][32 * kp + 4 * g]);
          const bf16x4 a1 = *reinterpret_cast<const bf16x4*>(&s_v[16 * ht + r][32 * kp + 16 + 4 * g]);
          const bf16x8 a = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
          for (int tt = 0; tt < 2; ++tt) o[ht][tt] = mfma32(a, p[kp][tt], o[ht][tt]);
        }
    }
  };
  auto total = [&](float v) {  // over the four lanes that share a query
    v += __shfl_xor(v, 16);
    return v + __shfl_xor(v, 32);
  };

  // a query tile never crosses a window (a multiple of 64): keys from its start to the last query
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    m[tt] = -INFINITY;
    l[tt] = 0.f;
#pragma unroll
    for (int ht = 0; ht < 4; ++ht) o[ht][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int start = t0 - t0 % window;
  attend(Keys{k + kv_row * T * kHd, vt + kv_row * kHd * Tp, T, Tp}, start, min(t0 + kQTile, T), t0);
  f32x4 y[4][2];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const float inv = 1.0f / total(l[tt]);
#pragma unroll
    for (int ht = 0; ht < 4; ++ht) y[ht][tt] = o[ht][tt] * inv;
  }
  // landmarks of the chunks before this one (a chunk is a multiple of 32), beside a null slot of
  // score 0 and value 0
  const int seen = min(t0 / land_chunk, n_land);
  if (seen > 0) {
    const float x = mix16 ? load_as<bf16_bits>(static_cast<const bf16_bits*>(mix)) : *static_cast<const float*>(mix);
    const float weight = 1.0f / (1.0f + expf(-x));
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      m[tt] = 0.f;
      l[tt] = g == 0 ? 1.f : 0.f;
#pragma unroll
      for (int ht = 0; ht < 4; ++ht) o[ht][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    attend(Keys{lk + kv_row * n_land * kHd, lvt + kv_row * kHd * land_tp, n_land, land_tp}, 0, seen, seen);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      const float inv = weight / total(l[tt]);
#pragma unroll
      for (int ht = 0; ht < 4; ++ht) y[ht][tt] += o[ht][tt] * inv;
    }
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const int t = t0 + 16 * tt + r;
    if (t >= T) continue;
    bf16_bits* dst = out + (((int64_t)b * T + t) * kv_heads * REP + h) * kHd + 4 * g;
#pragma unroll
    for (int ht = 0; ht < 4; ++ht) {
      u32x2 w;
      w.x = bf16_pair(y[ht][tt][0], y[ht][tt][1]);
      w.y = bf16_pair(y[ht][tt][2], y[ht][tt][3]);
      *reinterpret_cast<u32x2*>(dst + 16 * ht) = w;
    }
  }
}

// ------------------------------------------------------------------------------------------
// The decode state after a prompt, zeros included, in one launch (nine of the stock ops): window
// slots 0 .. n - 1 from the rows after the last whole window (keys transposed), landmark slots
// 1 .. full, per (sequence, KV head) in blockIdx.y.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fl_refresh_state_kernel(
    const bf16_bits* __restrict__ k, const bf16_bits* __restrict__ kv, const bf16_bits* __restrict__ lk,
    const bf16_bits* __restrict__ lkv, int T, int heads, int window, int full, int slots,
    bf16_bits* __restrict__ kt, bf16_bits* __restrict__ v, bf16_bits* __restrict__ lkt,
    bf16_bits* __restrict__ lv) {
  const int64_t bh = blockIdx.y, b = bh / heads, h = bh - b * heads;
  const int g0 = T / window * window, n = T - g0, row = 2 * heads * kHd;
  const int wn = window * kHd, ln = slots * kHd;
  int i = blockIdx.x * 256 + threadIdx.x;
  if (i < wn) {
    const int d = i / window, s = i - d * window;
    kt[bh * wn + i] = s < n ? k[(bh * T + g0 + s) * kHd + d] : 0;
    return;
  }
  i -= wn;
  if (i < wn) {
    const int s = i / kHd, d = i - s * kHd;
    v[bh * wn + i] = s < n ? kv[(b * T + g0 + s) * row + (heads + h) * kHd + d] : 0;
    return;
  }
  i -= wn;
  if (i < ln) {
    const int d = i / slots, s = i - d * slots - 1;
    lkt[bh * ln + i] = s >= 0 && s < full ? lk[(bh * full + s) * kHd + d] : 0;
    return;
  }
  i -= ln;
  if (i < ln) {
    const int s = i / kHd - 1, d = i - (s + 1) * kHd;
    lv[bh * ln + i] = s >= 0 && s < full ? lkv[(b * full + s) * row + (heads + h) * kHd + d] : 0;
  }
}

// ------------------------------------------------------------------------------------------
// Mean latent of every completed chunk (fp32 sum, rounded to bf16), and the fp32 sum of the rows
// after the last one (the decode state; zeros when there are none). One block per (chunk, sequence,
// 256 columns): 32 column groups of 16 bytes x 8 row groups.
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fl_latent_mean_kernel(const bf16_bits* __restrict__ latent, int64_t sb,
                                                             int64_t st, int T, int chunk, int n_full, int width,
                                                             bf16_bits* __restrict__ mean,
                                                             float* __restrict__ tail) {
  __shared__ float s_sum[8][256 + 8];
  const int j = blockIdx.x, b = blockIdx.y, cg = threadIdx.x & 31, rg = threadIdx.x >> 5;
  const int c = (blockIdx.z * 32 + cg) * 8;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const int end = min((j + 1) * chunk, T);
  if (c < width) {
    const bf16_bits* p = latent + b * sb + c;
#pragma unroll 4
    for (int t = j * chunk + rg; t < end; t += 8) {
      float v[8];
      Vec<bf16_bits, 8>::load(p + (int64_t)t * st, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += v[e];
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) s_sum[rg][cg * 8 + e] = acc[e];
  __syncthreads();
  const int col = blockIdx.z * 256 + threadIdx.x;
  if (col >= width) return;
  float t = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) t += s_sum[i][threadIdx.x];
  if (j < n_full) {
    mean[((int64_t)b * n_full + j) * width + col] = (bf16_bits)bf16_bits_of(t / (float)chunk);
  } else {
    tail[(int64_t)b * width + col] = t;
  }
}

// ------------------------------------------------------------------------------------------
// out = x rsqrt(mean x^2 + eps) w, bf16, one wave per row, 16 bytes per lane and access. Bound by
// memory. Rows 8,192 x 1,024 (34 MB): 7.3 us, 4.6 TB/s; the stock
// kernel takes 13.6 us.
// ------------------------------------------------------------------------------------------
template <int NV>
__global__ __launch_bounds__(256) void fl_rms_norm_kernel(const bf16_bits* __restrict__ x, int64_t rows, int dim,
                                                          const void* __restrict__ w, int w16, float eps,
                                                          float inv_dim, bf16_bits* __restrict__ out) {
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  const bf16_bits* p = x + row * dim;
  float v[NV][8], acc = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c < dim) {
      Vec<bf16_bits, 8>::load(p + c, v[i]);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fmaf(v[i][j], v[i][j], acc);
    }
  }
  const float scale = rsqrtf(fmaf(wave_sum(acc), inv_dim, eps));
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c < dim) {
      float ww[8];
      if (w16) Vec<bf16_bits, 8>::load(static_cast<const bf16_bits*>(w) + c, ww);
      else Vec<float, 8>::load(static_cast<const float*>(w) + c, ww);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[i][j] = (v[i][j] * scale) * ww[j];
      Vec<bf16_bits, 8>::store(out + row * dim + c, v[i]);
    }
  }
}

inline int64_t pad64(int64_t n) { return cdiv(n, 64) * 64; }

struct AttnLayout {
  size_t k, vt, lk, lvt, bytes;
};

AttnLayout attn_layout(int64_t B, int64_t T, int64_t kv_heads, int64_t n_land) {
  AttnLayout a;
  a.k = 0;
  a.vt = a.k + (size_t)(B * kv_heads * T * kHd) * 2;
  a.lk = a.vt + (size_t)(B * kv_heads * kHd * pad64(T)) * 2;
  a.lvt = a.lk + (size_t)(B * kv_heads * n_land * kHd) * 2;
  a.bytes = a.lvt + (size_t)(B * kv_heads * kHd * pad64(n_land)) * 2;
  return a;
}

}  // namespace

extern "C" {

size_t fl_refresh_workspace_bytes(int64_t B, int64_t T, int64_t kv_heads, int64_t n_landmarks) {
  if (B <= 0 || T <= 0 || kv_heads <= 0 || n_landmarks < 0) return 0;
  return attn_layout(B, T, kv_heads, n_landmarks).bytes;
}

int fl_refresh_attention(const void* q, int64_t q_stride_b, int64_t q_stride_t, const void* kv,
                         const void* landmark_kv, int64_t B, int64_t T, int64_t q_heads, int64_t kv_heads,
                         int64_t window, int64_t n_landmarks, int64_t landmark_chunk, const void* cos,
                         const void* sin, const void* mix_logit, int mix_dtype, void* out, void* workspace,
                         size_t workspace_bytes, void* stream) {
  if (!dtype_ok(mix_dtype)) return FL_ERR_DTYPE;
  if (B <= 0 || T <= 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads || B > 65535 || kv_heads > 4096 ||
      T > ((int64_t)1 << 28) || B * kv_heads * pad64(T) > ((int64_t)1 << 40))
    return FL_ERR_INVALID_ARGUMENT;
  const int64_t rep = q_heads / kv_heads;
  if (rep != 1 && rep != 2 && rep != 4 && rep != 8) return FL_ERR_INVALID_ARGUMENT;
  if (window <= 0 || window % 64 || window > ((int64_t)1 << 28) || landmark_chunk <= 0 || landmark_chunk % 32 ||
      landmark_chunk > ((int64_t)1 << 28) || n_landmarks < 0 || n_landmarks > T / landmark_chunk)
    return FL_ERR_INVALID_ARGUMENT;
  if (q_stride_t < q_heads * kHd || q_stride_b < 0 || q_stride_t % 8 || q_stride_b % 8 ||
      (B > 1 && q_stride_b < (T - 1) * q_stride_t + q_heads * kHd))
    return FL_ERR_INVALID_ARGUMENT;
  if (!q || !kv || !cos || !sin || !mix_logit || !out || (n_landmarks > 0 && !landmark_kv))
    return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(q, 16) || !aligned(kv, 16) || !aligned(landmark_kv, 16) || !aligned(cos, 16) || !aligned(sin, 16) ||
      !aligned(out, 16) || !aligned(mix_logit, esize(mix_dtype)))
    return FL_ERR_INVALID_ARGUMENT;
  const AttnLayout lay = attn_layout(B, T, kv_heads, n_landmarks);
  if (!workspace || workspace_bytes < lay.bytes) return FL_ERR_WORKSPACE;
  if (!aligned(workspace, 16)) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  bf16_bits *k = reinterpret_cast<bf16_bits*>(ws + lay.k), *vt = reinterpret_cast<bf16_bits*>(ws + lay.vt);
  bf16_bits *lk = reinterpret_cast<bf16_bits*>(ws + lay.lk), *lvt = reinterpret_cast<bf16_bits*>(ws + lay.lvt);
  const bf16_bits *c = static_cast<const bf16_bits*>(cos), *sn = static_cast<const bf16_bits*>(sin);
  const int64_t row = 2 * kv_heads * kHd;
  fl_rope_kv_kernel<<<dim3((unsigned)cdiv(T, 64), (unsigned)kv_heads, (unsigned)B), 256, 0, s>>>(
      static_cast<const bf16_bits*>(kv), T * row, row, (int)T, (int)pad64(T), (int)kv_heads, 0, 1, c, sn, k, vt);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_status(e);
  if (n_landmarks > 0) {
    fl_rope_kv_kernel<<<dim3((unsigned)cdiv(n_landmarks, 64), (unsigned)kv_heads, (unsigned)B), 256, 0, s>>>(
        static_cast<const bf16_bits*>(landmark_kv), n_landmarks * row, row, (int)n_landmarks,
        (int)pad64(n_landmarks), (int)kv_heads, (int)landmark_chunk - 1, (int)landmark_chunk, c, sn, lk, lvt);
    e = hipGetLastError();
    if (e != hipSuccess) return hip_status(e);
  }
  const dim3 grid((unsigned)cdiv(T, kQTile), (unsigned)kv_heads, (unsigned)B);
#define FL_ATTN(R)                                                                                        \
  fl_window_attention_kernel<R><<<grid, 64 * R, 0, s>>>(                                                  \
      static_cast<const bf16_bits*>(q), q_stride_b, q_stride_t, (int)T, (int)pad64(T), (int)kv_heads,     \
      (int)window, k, vt, (int)n_landmarks, (int)pad64(n_landmarks), (int)landmark_chunk, lk, lvt, c, sn, \
      mix_logit, mix_dtype == FL_DTYPE_BF16, static_cast<bf16_bits*>(out))
  switch (rep) {
    case 1: FL_ATTN(1); break;
    case 2: FL_ATTN(2); break;
    case 4: FL_ATTN(4); break;
    default: FL_ATTN(8); break;
  }
#undef FL_ATTN
  return hip_status(hipGetLastError());
}

int fl_refresh_state(const void* workspace, const void* kv, const void* landmark_kv, int64_t B, int64_t T,
                     int64_t kv_heads, int64_t window, int64_t n_landmarks, int64_t slots, void* kt, void* v,
                     void* lkt, void* lv, void* stream) {
  if (B <= 0 || T <= 0 || kv_heads <= 0 || B * kv_heads > 65535 || T > ((int64_t)1 << 28) || window <= 0 ||
      window > ((int64_t)1 << 20) || n_landmarks < 0 || slots <= n_landmarks || slots > ((int64_t)1 << 20))
    return FL_ERR_INVALID_ARGUMENT;
  if (!workspace || !kv || !kt || !v || !lkt || !lv || (n_landmarks > 0 && !landmark_kv)) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(workspace, 16) || !aligned(kv, 2) || !aligned(landmark_kv, 2) || !aligned(kt, 2) || !aligned(v, 2) ||
      !aligned(lkt, 2) || !aligned(lv, 2))
    return FL_ERR_INVALID_ARGUMENT;
  const AttnLayout lay = attn_layout(B, T, kv_heads, n_landmarks);
  const char* ws = static_cast<const char*>(workspace);
  fl_refresh_state_kernel<<<dim3((unsigned)cdiv(2 * (window + slots) * kHd, 256), (unsigned)(B * kv_heads)), 256, 0,
                            static_cast<hipStream_t>(stream)>>>(
      reinterpret_cast<const bf16_bits*>(ws + lay.k), static_cast<const bf16_bits*>(kv),
      reinterpret_cast<const bf16_bits*>(ws + lay.lk), static_cast<const bf16_bits*>(landmark_kv), (int)T,
      (int)kv_heads, (int)window, (int)n_landmarks, (int)slots, static_cast<bf16_bits*>(kt),
      static_cast<bf16_bits*>(v), static_cast<bf16_bits*>(lkt), static_cast<bf16_bits*>(lv));
  return hip_status(hipGetLastError());
}

int fl_latent_mean(const void* latent, int64_t stride_b, int64_t stride_t, int64_t B, int64_t T, int64_t chunk,
                   int64_t width, void* mean, float* tail, void* stream) {
  if (B <= 0 || T <= 0 || chunk <= 0 || width <= 0 || width % 8 || B > 65535 || T > ((int64_t)1 << 28) ||
      chunk > ((int64_t)1 << 28) || width > ((int64_t)1 << 16))
    return FL_ERR_INVALID_ARGUMENT;
  if (stride_t < width || stride_t % 8 || stride_b < 0 || stride_b % 8 ||
      (B > 1 && stride_b < (T - 1) * stride_t + width))
    return FL_ERR_INVALID_ARGUMENT;
  const int64_t n_full = T / chunk;
  if (!latent || !tail || (n_full > 0 && !mean)) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(latent, 16) || !aligned(mean, 2) || !aligned(tail, 4)) return FL_ERR_INVALID_ARGUMENT;
  fl_latent_mean_kernel<<<dim3((unsigned)(n_full + 1), (unsigned)B, (unsigned)cdiv(width, 256)), 256, 0,
                          static_cast<hipStream_t>(stream)>>>(
      static_cast<const bf16_bits*>(latent), stride_b, stride_t, (int)T, (int)chunk, (int)n_full, (int)width,
      static_cast<bf16_bits*>(mean), tail);
  return hip_status(hipGetLastError());
}

int fl_rms_norm(const void* x, int64_t rows, int64_t dim, const void* weight, int w_dtype, float eps, void* out,
                void* stream) {
  if (!dtype_ok(w_dtype)) return FL_ERR_DTYPE;
  if (rows <= 0 || rows > ((int64_t)1 << 31) - 1 || dim <= 0 || dim % 8 || dim > 4096) return FL_ERR_INVALID_ARGUMENT;
  if (!x || !weight || !out || !(eps >= 0.f)) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(x, 16) || !aligned(weight, 16) || !aligned(out, 16)) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // one row per block while the rows are few, to spread them over the CUs. us, one | four rows a block: dim 1,024,
  // 64 rows 2.5 | 2.7, 512 2.8 | 2.8, 4,096 4.6 | 4.2, 16,384 12.0 | 12.4; dim 512, 16,384 rows 7.2 | 5.8
  const unsigned waves = rows >= 4096 ? 4 : 1;
  const unsigned blocks = (unsigned)cdiv(rows, waves);
  const float inv = (float)(1.0 / (double)dim);
  const bf16_bits* xp = static_cast<const bf16_bits*>(x);
  bf16_bits* o = static_cast<bf16_bits*>(out);
  const int w16 = w_dtype == FL_DTYPE_BF16;
  if (dim <= 1024) {
    fl_rms_norm_kernel<2><<<blocks, waves * 64, 0, s>>>(xp, rows, (int)dim, weight, w16, eps, inv, o);
  } else {
    fl_rms_norm_kernel<8><<<blocks, waves * 64, 0, s>>>(xp, rows, (int)dim, weight, w16, eps, inv, o);
  }
  return hip_status(hipGetLastError());
}

}  // extern "C"
