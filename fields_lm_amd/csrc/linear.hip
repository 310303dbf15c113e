// linear.hip — the Field block's products for a few rows (one token of a decode batch), bf16 with
// fp32 sums, each with the elementwise work around it (reference: src/fields_official/reference/
// field_only_v4_chunked_triton_wiki100.py:1167-1221; single-token steps have no counterpart there).
//
// A decode step reads every weight once: 26 MB per block at dim 1,024, 5 us at the rate of a large
// copy. A block of the grid owns 16 output columns of 16 rows (32 where rows are many); its waves split the depth, so each
// wave's part is a few 16-byte loads per lane that are all in flight together, and the partial sums
// meet in LDS in a fixed order. More rows per block read the weights fewer times from L2, but put the
// reading of the rows on fewer CUs, each bound by its loads in flight: 64 rows in one tile took 56 us
// for the five launches, in two 44, in four 40. What used to be separate launches rides along:
//   in:    [write_proj | gate_proj] from the two layers' own weights
//   out:   out_proj, then x + out * sigmoid(gate)
//   up:    RMSNorm of its input (the row's scale is applied to the sums, the weight to the operand),
//          gate and up columns in one block, then silu(gate) * up
//   down:  the FFN's output product, added to the residual
// 64 rows, dim 1,024, hidden 2,528: 41.1 us of kernels with the weights in the Infinity Cache (in 9.3, norm
// 3.7, out 9.0, up 13.5, down 5.7) and 42 us in a graph over 12 blocks' cold weights, where the library's
// products and separate launches take 58 us; one row 27 us cold against 56.
#include "fl_common.h"

namespace {

using namespace fl;

enum Epilogue { kBias, kGatedResidual, kNormSwiglu, kResidual };

struct LinearArgs {
  const bf16_bits* x;   // [M, K], rows x_stride apart
  int64_t x_stride;
  const bf16_bits* w;   // [n1, K]; columns from n1 on (kBias: the second layer; kNormSwiglu: up) in w2
  const bf16_bits* w2;
  const bf16_bits* b;   // [n1] or NULL
  const bf16_bits* b2;
  int M, N, K, n1;
  const bf16_bits* gate;  // kGatedResidual: gate_pre, rows gate_stride apart
  int64_t gate_stride;
  const bf16_bits* res;   // kGatedResidual, kResidual: [M, N]
  const void* norm_w;     // kNormSwiglu: [K]
  int norm_w16;
  float eps;
  bf16_bits* out;         // [M, N]
};

constexpr int kSlots = 8;    // partial sums kept in LDS (16 waves fold once before)
constexpr int kAccRow = 20;  // floats per row of 16 columns

// 16 MT rows, W waves, G depth steps of 32 loaded together
template <int EPI, int W, int G, int MT>
__global__ __launch_bounds__(W * 64, W / 4) void fl_linear_rows_kernel(LinearArgs a) {
  constexpr int S = EPI == kNormSwiglu ? 2 : 1;  // column sets: gate and up share the rows' operand
  __shared__ float s_acc[kSlots][S][16 * MT][kAccRow], s_sq[W][16 * MT];
  const int tid = threadIdx.x, lane = tid & 63, wave = uniform(tid >> 6), r = lane & 15, k8 = 8 * (lane >> 4);
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
  if (n0 >= a.N) return;  // the grid's width is rounded up
  const int n = min(n0 + r, a.N - 1);
  const bf16_bits* wp[S];
  if constexpr (S == 2) {
    wp[0] = a.w + (int64_t)n * a.K;
    wp[1] = a.w2 + (int64_t)n * a.K;
  } else {
    wp[0] = n < a.n1 ? a.w + (int64_t)n * a.K : a.w2 + (int64_t)(n - a.n1) * a.K;
  }
  const bf16_bits* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = a.x + (int64_t)min(m0 + 16 * t + r, a.M - 1) * a.x_stride;

  const int steps = (a.K + 31) / 32, per = (steps + W - 1) / W;
  const int first = min(wave * per, steps), last = min(first + per, steps);
  f32x4 acc[S][MT];
  float sq[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    sq[t] = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const u32x4 zero = {0u, 0u, 0u, 0u};
  for (int step = first; step < last; step += G) {
    u32x4 wf[G][S], xf[G][MT];
    float nw[G][EPI == kNormSwiglu ? 8 : 1];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int k = (step + i) * 32 + k8;
      const bool in = step + i < last && k < a.K;  // a whole vector or none: K is a multiple of 8
      const int kc = in ? k : 0;
#pragma unroll
      for (int s = 0; s < S; ++s) {
        wf[i][s] = *reinterpret_cast<const u32x4*>(wp[s] + kc);
        if (!in) wf[i][s] = zero;
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        xf[i][t] = *reinterpret_cast<const u32x4*>(xp[t] + kc);
        if (!in) xf[i][t] = zero;
      }
      if constexpr (EPI == kNormSwiglu) {
        if (a.norm_w16) Vec<bf16_bits, 8>::load(static_cast<const bf16_bits*>(a.norm_w) + kc, nw[i]);
        else Vec<float, 8>::load(static_cast<const float*>(a.norm_w) + kc, nw[i]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);  // every load of the group is issued before the first product
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        u32x4 xv = xf[i][t];
        if constexpr (EPI == kNormSwiglu) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float lo = bf16_lo(xv[e]), hi = bf16_hi(xv[e]);
            sq[t] = fmaf(lo, lo, fmaf(hi, hi, sq[t]));
            xv[e] = bf16_pair(lo * nw[i][2 * e], hi * nw[i][2 * e + 1]);
          }
        }
#pragma unroll
        for (int s = 0; s < S; ++s)
          acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[i][s]),
                                                              __builtin_bit_cast(bf16x8, xv), acc[s][t], 0, 0, 0);
      }
  }
  // lane: columns 4 (lane / 16) .. + 3 of row r
  if constexpr (EPI == kNormSwiglu) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      sq[t] += __shfl_xor(sq[t], 16);
      sq[t] += __shfl_xor(sq[t], 32);
      if (lane < 16) s_sq[wave][16 * t + r] = sq[t];
    }
  }
  auto put = [&](int slot) {
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < MT; ++t) *reinterpret_cast<f32x4*>(&s_acc[slot][s][16 * t + r][k8 / 2]) = acc[s][t];
  };
  if constexpr (W > kSlots) {
    static_assert(W == 2 * kSlots, "one fold");
    if (wave >= kSlots) put(wave - kSlots);
    __syncthreads();
    if (wave < kSlots) {
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[s][t] += *reinterpret_cast<const f32x4*>(&s_acc[wave][s][16 * t + r][k8 / 2]);
      put(wave);  // its own slot, read by itself alone
    }
  } else {
    put(wave);
  }
  __syncthreads();
  if (tid < MT * 16 * 8) {
    const int row = tid >> 3, c = 2 * (tid & 7), m = m0 + row;
    if (m >= a.M) return;
    float v[S][2];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      v[s][0] = v[s][1] = 0.f;
#pragma unroll
      for (int u = 0; u < (W < kSlots ? W : kSlots); ++u) {
        v[s][0] += s_acc[u][s][row][c];
        v[s][1] += s_acc[u][s][row][c + 1];
      }
    }
    float scale = 1.f;
    if constexpr (EPI == kNormSwiglu) {
      float t = 0.f;
#pragma unroll
      for (int u = 0; u < W; ++u) t += s_sq[u][row];
      scale = rsqrtf(t / (float)a.K + a.eps);
    }
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int col = n0 + c + e;
      if (col >= a.N) break;
      const int64_t at = (int64_t)m * a.N + col;
      float o = v[0][e];
      if constexpr (EPI == kBias || EPI == kGatedResidual) {
        const bf16_bits* bias = col < a.n1 ? a.b : a.b2;
        if (bias != nullptr) o += load_as<bf16_bits>(bias + (col < a.n1 ? col : col - a.n1));
      }
      if constexpr (EPI == kGatedResidual) {
        const float g = load_as<bf16_bits>(a.gate + (int64_t)m * a.gate_stride + col);
        const float sg = bf16_round(sigmoid_bf16(g));
        o = load_as<bf16_bits>(a.res + at) + bf16_round(bf16_round(o) * sg);
      } else if constexpr (EPI == kNormSwiglu) {
        o = bf16_round(silu_precise(bf16_round(o * scale))) * bf16_round(v[1][e] * scale);
      } else if constexpr (EPI == kResidual) {
        o += load_as<bf16_bits>(a.res + at);
      }
      a.out[at] = (bf16_bits)bf16_bits_of(o);
    }
  }
}

// 16 columns and 16 MT rows a block
template <int EPI, int MT>
void launch_tiles(const LinearArgs& a, hipStream_t s) {
  // Row tiles of one column tile lie a multiple of 8 blocks apart: on one XCD, whose L2 then holds
  // their common weights.
  const dim3 grid((unsigned)(cdiv(cdiv(a.N, 16), 8) * 8), (unsigned)cdiv(a.M, 16 * MT));
  // 8 waves reach a depth of 1,024 (1,280 with a group of 5) with one group of loads each; deeper products
  // take 16.
  if constexpr (EPI == kNormSwiglu) {
    fl_linear_rows_kernel<EPI, 8, 4, MT><<<grid, 512, 0, s>>>(a);
  } else if (a.K <= 1024) {
    fl_linear_rows_kernel<EPI, 8, 4, MT><<<grid, 512, 0, s>>>(a);
  } else if (a.K <= 1280) {
    fl_linear_rows_kernel<EPI, 8, 5, MT><<<grid, 512, 0, s>>>(a);
  } else {
    fl_linear_rows_kernel<EPI, 16, 5, MT><<<grid, 1024, 0, s>>>(a);
  }
}

template <int EPI>
int launch_linear(const LinearArgs& a, bool two, hipStream_t s) {
  if (two) launch_tiles<EPI, 2>(a, s);
  else launch_tiles<EPI, 1>(a, s);
  return hip_status(hipGetLastError());
}

constexpr int64_t kMaxRows = 128;

bool vec_ok(const void* p) { return p != nullptr && aligned(p, 16); }

}  // namespace

extern "C" {

int fl_block_step(const void* x, int64_t rows, int64_t dim, int64_t hidden, const void* write_w, const void* write_b,
                  const void* gate_w, const void* gate_b, const float* tr, const float* ti, const float* gamma,
                  float* state, const float* read_norm_w, float read_eps, const void* out_w, const void* out_b,
                  const void* ff_norm_w, int ff_norm_dtype, float ff_eps, const void* up_w, const void* down_w,
                  void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (!dtype_ok(ff_norm_dtype)) return FL_ERR_DTYPE;
  if (rows <= 0 || rows > kMaxRows || dim <= 0 || dim % 8 || dim > 8192 || hidden <= 0 || hidden % 8 || hidden > 65536)
    return FL_ERR_INVALID_ARGUMENT;
  if (!vec_ok(x) || !vec_ok(write_w) || !vec_ok(gate_w) || !vec_ok(out_w) || !vec_ok(up_w) || !vec_ok(down_w) ||
      !vec_ok(ff_norm_w) || !vec_ok(out) || !tr || !ti || !gamma || !state || !read_norm_w ||
      !aligned(write_b, 2) || !aligned(gate_b, 2) || !aligned(out_b, 2) || !(read_eps >= 0.f) || !(ff_eps >= 0.f))
    return FL_ERR_INVALID_ARGUMENT;
  if (!workspace || workspace_bytes < fl_block_step_workspace_bytes(rows, dim, hidden)) return FL_ERR_WORKSPACE;
  if (!aligned(workspace, 16)) return FL_ERR_INVALID_ARGUMENT;
  const int64_t C = dim / 2, wide = 3 * C + dim;
  bf16_bits* y = static_cast<bf16_bits*>(workspace);                    // [rows, raw 3C | gate dim]
  bf16_bits* normed = y + cdiv(rows * wide, 8) * 8;                     // [rows, 2 dim]
  bf16_bits* x1 = normed + rows * 2 * dim;                              // [rows, dim]
  bf16_bits* act = x1 + rows * dim;                                     // [rows, hidden]
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto bf = [](const void* p) { return static_cast<const bf16_bits*>(p); };
  const int M = (int)rows, D = (int)dim, H = (int)hidden;
  // Two row tiles a block once the blocks of one no longer fit the chip side by side. us in a graph over cold
  // weights, one | two: dim 512: 96 rows 33.1 | 34.3; 768: 80 rows 39.8 | 43.2, 96 48.3 | 44.9; 1,024: 64 rows
  // 42.3 | 47.5, 80 54.1 | 45.8, 128 60.1 | 55.5; 1,152: 48 rows 57.2 | 60.3, 64 70.0 | 65.3; 1,280: 32 rows
  // 51.9 | 56.4, 64 76.4 | 66.9, 128 113.7 | 105.5; 2,048: 32 rows 76.9 | 90.4, 48 104.2 | 94.8
  const bool two = rows * dim > 65536;

  LinearArgs in{};
  in.x = bf(x); in.x_stride = dim; in.w = bf(write_w); in.w2 = bf(gate_w); in.b = bf(write_b); in.b2 = bf(gate_b);
  in.M = M; in.N = (int)wide; in.K = D; in.n1 = (int)(3 * C); in.out = y;
  int rc = launch_linear<kBias>(in, two, s);
  if (rc != FL_OK) return rc;

  rc = fl_decode_norm_step(y, FL_DTYPE_BF16, rows, C, wide, tr, ti, gamma, state, read_norm_w, read_eps, normed,
                           FL_DTYPE_BF16, stream);
  if (rc != FL_OK) return rc;

  LinearArgs o{};
  o.x = normed; o.x_stride = 2 * dim; o.w = o.w2 = bf(out_w); o.b = o.b2 = bf(out_b);
  o.M = M; o.N = D; o.K = 2 * D; o.n1 = D; o.gate = y + 3 * C; o.gate_stride = wide; o.res = bf(x); o.out = x1;
  rc = launch_linear<kGatedResidual>(o, two, s);
  if (rc != FL_OK) return rc;

  LinearArgs u{};
  u.x = x1; u.x_stride = dim; u.w = bf(up_w); u.w2 = bf(up_w) + hidden * dim;
  u.M = M; u.N = H; u.K = D; u.n1 = H; u.norm_w = ff_norm_w; u.norm_w16 = ff_norm_dtype == FL_DTYPE_BF16;
  u.eps = ff_eps; u.out = act;
  rc = launch_linear<kNormSwiglu>(u, two, s);
  if (rc != FL_OK) return rc;

  LinearArgs d{};
  d.x = act; d.x_stride = hidden; d.w = d.w2 = bf(down_w);
  d.M = M; d.N = D; d.K = H; d.n1 = D; d.res = x1; d.out = static_cast<bf16_bits*>(out);
  return launch_linear<kResidual>(d, two, s);
}

size_t fl_block_step_workspace_bytes(int64_t rows, int64_t dim, int64_t hidden) {
  if (rows <= 0 || dim <= 0 || hidden <= 0) return 0;
  return (size_t)(cdiv(rows * (dim / 2 * 3 + dim), 8) * 8 + rows * (3 * dim + hidden)) * 2;
}

}  // extern "C"
