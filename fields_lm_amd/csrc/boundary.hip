// boundary.hip — the softpatch mixer's boundary scan (reference: src/fields_official/reference/
// official_source/field_hybrid_attentionfree_qualification_v3.py:441-464,
// field_hybrid_speed_optimization_v6.py:318-338), on its own (fl_boundary_scan) and with the work
// around it (fl_softpatch_norm, fl_softpatch_scan).
#include "fl_common.h"

namespace {

using namespace fl;

// ------------------------------------------------------------------------------------------
//   s[b,t,r] = a[b,t] * s[b,t-1,r] + drive[b,t,r],   s[b,-1,:] = state_in or 0,
// the real-valued first-order recurrence that the reference runs through
// hierarchical_scan(a, drive, block=32) with a = (1 - boundary) broadcast over the rank.
// Block = (batch row, 64 channels), W waves; wave w owns steps [w*S, (w+1)*S). Pass 1 forms
// each wave's map (prod a, state from 0) over its steps, the waves' carries are composed in LDS,
// pass 2 re-runs from the carry and stores. Lane <-> channel, so each step is one coalesced
// row of loads and stores; a[b,t] is the same for the whole wave: the lanes hold 64 steps' values
// and each is read from its lane.
// Few blocks (B x R / 64), so bound by the latency of the wave's serial steps: rows are loaded kBatch
// at a time, ahead of the batch being applied (one load per step left each step waiting for
// memory). B=4, T=2,048, R=64: 64 us with a load per step, 28 us so.
// ------------------------------------------------------------------------------------------
constexpr int kBoundaryWaves = 16;
constexpr int kBatch = 32;

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}

// Steps [t0, t1) in order: `gate(t)` gives a lane its step's gate value (64 steps at a time), `row(t)`
// the lane's channel of row t, and `apply(gate_t, row_t, t)` takes them. The rows of the next batch are
// requested before a batch is applied, without a branch per row (past the end the last row again): with
// one, each load was waited for by itself.
template <typename Gate, typename Row, typename Apply>
__device__ __forceinline__ void walk(int t0, int t1, int lane, Gate gate, Row row, Apply apply) {
  if (t0 >= t1) return;
  float next[kBatch], g = 0.f;
#pragma unroll
  for (int i = 0; i < kBatch; ++i) next[i] = row(min(t0 + i, t1 - 1));
  for (int t = t0; t < t1; t += kBatch) {
    const int at = (t - t0) & 63;
    if (at == 0) g = gate(min(t + lane, t1 - 1));
    float v[kBatch];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) v[i] = next[i];
#pragma unroll
    for (int i = 0; i < kBatch; ++i) next[i] = row(min(t + kBatch + i, t1 - 1));
    if (t + kBatch <= t1) {
#pragma unroll
      for (int i = 0; i < kBatch; ++i) apply(lane_value(g, at + i), v[i], t + i);
    } else {
#pragma unroll
      for (int i = 0; i < kBatch; ++i)
        if (t + i < t1) apply(lane_value(g, at + i), v[i], t + i);
    }
  }
}

__global__ __launch_bounds__(kBoundaryWaves * 64) void fl_boundary_scan_kernel(
    const float* __restrict__ a, const float* __restrict__ drive, int T, int R,
    const float* __restrict__ state_in, float* __restrict__ state_out, float* __restrict__ out) {
  __shared__ float s_p[kBoundaryWaves][64], s_s[kBoundaryWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = uniform(threadIdx.x >> 6);
  const int b = blockIdx.x;
  const int r = blockIdx.y * 64 + lane;
  const bool ok = r < R;
  const int span = (T + kBoundaryWaves - 1) / kBoundaryWaves;
  const int t0 = min(wave * span, T), t1 = min(t0 + span, T);
  const float* ab = a + (int64_t)b * T;
  const float* db = drive + (int64_t)b * T * R + min(r, R - 1);
  float* ob = out + (int64_t)b * T * R + r;
  auto gate = [&](int t) { return ab[t]; };
  auto row = [&](int t) { return db[(int64_t)t * R]; };
  float p = 1.f, sv = 0.f;
  walk(t0, t1, lane, gate, row, [&](float at, float d, int) {
    sv = fmaf(at, sv, d);
    p *= at;
  });
  s_p[wave][lane] = p;
  s_s[wave][lane] = sv;
  __syncthreads();
  float c = (ok && state_in) ? state_in[(int64_t)b * R + r] : 0.f;
  for (int u = 0; u < wave; ++u) c = fmaf(s_p[u][lane], c, s_s[u][lane]);
  walk(t0, t1, lane, gate, row, [&](float at, float d, int t) {
    c = fmaf(at, c, d);
    if (ok) ob[(int64_t)t * R] = c;
  });
  if (ok && state_out && wave == kBoundaryWaves - 1) {
    // the last wave ends at T (or holds the composed carry when its span is empty)
    state_out[(int64_t)b * R + r] = c;
  }
}

// ------------------------------------------------------------------------------------------
// The same scan from the mixer's projections: boundary = clamp(sigmoid(score + 1.5 prior), 0.01, 0.99),
// a = 1 - boundary, drive = boundary z, and the output is what the up projection reads, [z | s] in
// bf16, so neither the gates nor the fp32 z, drive and state reach memory.
// A wave takes a chunk of 64 steps (its lanes' gates) and 64 channels, so that a few sequences still
// spread over many CUs: one launch forms every chunk's map (prod a, state from 0), the next folds the
// maps before its chunk, in order, and re-runs the chunk from there. B=4, T=2,048, R=64: 13.7 us for both
// launches, 28 us in one launch of a block per sequence.
// ------------------------------------------------------------------------------------------
struct SoftArgs {
  const bf16_bits* z;
  const bf16_bits* score;
  const float* prior;
  int T, R, n_chunks;
  float* maps;  // [B, R tiles, n_chunks, 65]: 64 states, then the gates' product
};

__device__ __forceinline__ float soft_gate(const SoftArgs& s, int64_t bt) {
  const float x = fmaf(1.5f, s.prior[bt], load_as<bf16_bits>(s.score + bt));
  const float g = 1.0f / (1.0f + expf(-x));
  return g != g ? g : fminf(fmaxf(g, 0.01f), 0.99f);
}

__global__ __launch_bounds__(256) void fl_softpatch_map_kernel(SoftArgs s) {
  const int lane = threadIdx.x & 63, chunk = blockIdx.x * 4 + uniform(threadIdx.x >> 6);
  if (chunk >= s.n_chunks) return;
  const int64_t b = blockIdx.z, bt = b * s.T;
  const int r = blockIdx.y * 64 + lane, t0 = chunk * 64, t1 = min(t0 + 64, s.T);
  const bf16_bits* zb = s.z + bt * s.R + min(r, s.R - 1);
  float p = 1.f, sv = 0.f;
  walk(t0, t1, lane, [&](int t) { return soft_gate(s, bt + t); },
       [&](int t) { return load_as<bf16_bits>(zb + (int64_t)t * s.R); },
       [&](float g, float zt, int) {
         const float at = 1.0f - g;
         sv = fmaf(at, sv, g * zt);
         p *= at;
       });
  float* m = s.maps + ((b * gridDim.y + blockIdx.y) * s.n_chunks + chunk) * 65;
  m[lane] = sv;
  if (lane == 0) m[64] = p;
}

__global__ __launch_bounds__(256) void fl_softpatch_scan_kernel(SoftArgs s, float* __restrict__ state_out,
                                                                bf16_bits* __restrict__ out) {
  const int lane = threadIdx.x & 63, chunk = blockIdx.x * 4 + uniform(threadIdx.x >> 6);
  if (chunk >= s.n_chunks) return;
  const int64_t b = blockIdx.z, bt = b * s.T;
  const int r = blockIdx.y * 64 + lane, t0 = chunk * 64, t1 = min(t0 + 64, s.T);
  const bool ok = r < s.R;
  const bf16_bits* zb = s.z + bt * s.R + min(r, s.R - 1);
  bf16_bits* ob = out + bt * 2 * s.R + r;
  const float* m = s.maps + (b * gridDim.y + blockIdx.y) * s.n_chunks * 65;
  float c = 0.f;
  if (chunk > 0)
    walk(0, chunk, lane, [&](int u) { return m[(int64_t)u * 65 + 64]; },
         [&](int u) { return m[(int64_t)u * 65 + lane]; }, [&](float p, float sv, int) { c = fmaf(p, c, sv); });
  walk(t0, t1, lane, [&](int t) { return soft_gate(s, bt + t); },
       [&](int t) { return load_as<bf16_bits>(zb + (int64_t)t * s.R); },
       [&](float g, float zt, int t) {
         c = fmaf(1.0f - g, c, g * zt);
         if (ok) {
           ob[(int64_t)t * 2 * s.R] = (bf16_bits)bf16_bits_of(zt);
           ob[(int64_t)t * 2 * s.R + s.R] = (bf16_bits)bf16_bits_of(c);
         }
       });
  if (ok && chunk == s.n_chunks - 1) state_out[b * s.R + r] = c;
}

// ------------------------------------------------------------------------------------------
// h = RMSNorm(x) and score = h . w_score + bias (h as rounded to bf16, fp32 sum, bf16 out): the row is
// in registers for the norm, so its one-column product costs no launch and no second read. One wave per
// row, bound by memory.
// ------------------------------------------------------------------------------------------
template <int NV>
__global__ __launch_bounds__(256) void fl_softpatch_norm_kernel(
    const bf16_bits* __restrict__ x, int64_t rows, int dim, const bf16_bits* __restrict__ w, float eps,
    float inv_dim, const bf16_bits* __restrict__ w_score, const bf16_bits* __restrict__ bias,
    bf16_bits* __restrict__ h, bf16_bits* __restrict__ score) {
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
  float dot = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c < dim) {
      float ww[8], ws[8];
      Vec<bf16_bits, 8>::load(w + c, ww);
      Vec<bf16_bits, 8>::load(w_score + c, ws);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] = (v[i][j] * scale) * ww[j];
        dot = fmaf(bf16_round(v[i][j]), ws[j], dot);
      }
      Vec<bf16_bits, 8>::store(h + row * dim + c, v[i]);
    }
  }
  dot = wave_sum(dot);
  if (lane == 0) score[row] = (bf16_bits)bf16_bits_of(dot + load_as<bf16_bits>(bias));
}

constexpr int64_t kMaxB = 65535, kMaxR = (int64_t)1 << 16, kMaxT = (int64_t)1 << 30;

}  // namespace

extern "C" {

int fl_boundary_scan(const float* a, const float* drive, int64_t B, int64_t T, int64_t R,
                     const float* state_in, float* state_out, float* out, void* stream) {
  if (B <= 0 || T <= 0 || R <= 0 || B > kMaxB || R > kMaxR || T > kMaxT)
    return FL_ERR_INVALID_ARGUMENT;
  if (T * R >= ((int64_t)1 << 40)) return FL_ERR_INVALID_ARGUMENT;
  if (!a || !drive || !out) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(a, 4) || !aligned(drive, 4) || !aligned(out, 4) ||
      (state_in && !aligned(state_in, 4)) || (state_out && !aligned(state_out, 4)))
    return FL_ERR_INVALID_ARGUMENT;
  const dim3 grid((unsigned)B, (unsigned)cdiv(R, 64));
  fl_boundary_scan_kernel<<<grid, kBoundaryWaves * 64, 0, static_cast<hipStream_t>(stream)>>>(
      a, drive, (int)T, (int)R, state_in, state_out, out);
  return hip_status(hipGetLastError());
}

int fl_softpatch_norm(const void* x, int64_t rows, int64_t dim, const void* weight, float eps, const void* w_score,
                      const void* bias, void* h, void* score, void* stream) {
  if (rows <= 0 || rows > ((int64_t)1 << 31) - 1 || dim <= 0 || dim % 8 || dim > 4096) return FL_ERR_INVALID_ARGUMENT;
  if (!x || !weight || !w_score || !bias || !h || !score || !(eps >= 0.f)) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(x, 16) || !aligned(weight, 16) || !aligned(w_score, 16) || !aligned(h, 16) || !aligned(bias, 2) ||
      !aligned(score, 2))
    return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  // one row per block while the rows are few, to spread them over the CUs. us, one | four rows a block: dim 1,024,
  // 64 rows 2.8 | 2.9, 512 3.0 | 3.1, 4,096 4.9 | 4.6, 16,384 12.5 | 12.9; dim 512, 16,384 rows 7.6 | 6.7
  const unsigned waves = rows >= 4096 ? 4 : 1;
  const unsigned blocks = (unsigned)cdiv(rows, waves);
  const float inv = (float)(1.0 / (double)dim);
#define FL_SN(NV)                                                                                            \
  fl_softpatch_norm_kernel<NV><<<blocks, waves * 64, 0, s>>>(                                                \
      static_cast<const bf16_bits*>(x), rows, (int)dim, static_cast<const bf16_bits*>(weight), eps, inv,     \
      static_cast<const bf16_bits*>(w_score), static_cast<const bf16_bits*>(bias), static_cast<bf16_bits*>(h), \
      static_cast<bf16_bits*>(score))
  if (dim <= 1024) {
    FL_SN(2);
  } else {
    FL_SN(8);
  }
#undef FL_SN
  return hip_status(hipGetLastError());
}

size_t fl_softpatch_workspace_bytes(int64_t B, int64_t T, int64_t R) {
  if (B <= 0 || T <= 0 || R <= 0) return 0;
  return (size_t)(B * cdiv(R, 64) * cdiv(T, 64)) * 65 * 4;
}

int fl_softpatch_scan(const void* z, const void* score, const float* prior, int64_t B, int64_t T, int64_t R,
                      float* state_out, void* out, void* workspace, size_t workspace_bytes, void* stream) {
  if (B <= 0 || T <= 0 || R <= 0 || B > kMaxB || R > kMaxR || T > kMaxT || T * R >= ((int64_t)1 << 39))
    return FL_ERR_INVALID_ARGUMENT;
  if (!z || !score || !prior || !state_out || !out) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(z, 2) || !aligned(score, 2) || !aligned(prior, 4) || !aligned(state_out, 4) || !aligned(out, 2))
    return FL_ERR_INVALID_ARGUMENT;
  if (!workspace || workspace_bytes < fl_softpatch_workspace_bytes(B, T, R)) return FL_ERR_WORKSPACE;
  if (!aligned(workspace, 4)) return FL_ERR_INVALID_ARGUMENT;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int n_chunks = (int)cdiv(T, 64);
  const SoftArgs args{static_cast<const bf16_bits*>(z), static_cast<const bf16_bits*>(score), prior, (int)T, (int)R,
                      n_chunks, static_cast<float*>(workspace)};
  const dim3 grid((unsigned)cdiv(n_chunks, 4), (unsigned)cdiv(R, 64), (unsigned)B);
  if (n_chunks > 1) {
    fl_softpatch_map_kernel<<<grid, 256, 0, s>>>(args);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_status(e);
  }
  fl_softpatch_scan_kernel<<<grid, 256, 0, s>>>(args, state_out, static_cast<bf16_bits*>(out));
  return hip_status(hipGetLastError());
}

}  // extern "C"
