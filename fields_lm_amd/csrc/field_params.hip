// field_params.hip — the Field mixer's transition parameters in one launch (reference:
// src/fields_official/reference/field_only_v4_chunked_triton_wiki100.py, "canon", 1169-1173).
//
// Built with -ffp-contract=on (the other sources: fast), which leaves products and sums of separate
// statements, and the exponential's own arithmetic, rounded as the stock ops round them: under fast,
// 1.6 % of the radii differed in their last bit.
#include "fl_common.h"

#pragma clang fp contract(off)

namespace {

using namespace fl;

// ------------------------------------------------------------------------------------------
// Transition parameters (canon:1169-1173): radius = clamp(sigmoid(radius_logit), 0.5, 0.99995),
// tr = radius cos(theta), ti = radius sin(theta), gamma = sqrt(max(1 - radius^2, 1e-4)); and a
// bf16 norm weight widened to fp32. Bit for bit the stock ops' values. A few KB, bound by the launch: one launch where the stock ops
// take twelve of 3.5-4.3 us each (C = 512: 4.2 us against 45 us).
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void fl_field_params_kernel(
    const float* __restrict__ radius_logit, const float* __restrict__ theta, int C,
    const bf16_bits* __restrict__ w16, int n_w, float* __restrict__ tr, float* __restrict__ ti,
    float* __restrict__ gamma, float* __restrict__ w32) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < C) {
    const float sg = 1.0f / (1.0f + expf(-radius_logit[i]));
    // a NaN logit stays NaN, as through the stock clamp
    const float r = sg != sg ? sg : fminf(fmaxf(sg, 0.50f), 0.99995f);
    const float th = theta[i];
    tr[i] = r * cosf(th);
    ti[i] = r * sinf(th);
    const float sq = r * r;
    const float d = 1.0f - sq;
    gamma[i] = d != d ? d : sqrtf(fmaxf(d, 1e-4f));
  }
  if (i < n_w) w32[i] = __uint_as_float((uint32_t)w16[i] << 16);
}

}  // namespace

extern "C" {

int fl_field_params(const float* radius_logit, const float* theta, int64_t C, const void* weight16,
                    int64_t n_weight, float* tr, float* ti, float* gamma, float* weight32,
                    void* stream) {
  if (C <= 0 || C > ((int64_t)1 << 24) || n_weight < 0 || n_weight > ((int64_t)1 << 26))
    return FL_ERR_INVALID_ARGUMENT;
  if (!radius_logit || !theta || !tr || !ti || !gamma) return FL_ERR_INVALID_ARGUMENT;
  if (n_weight > 0 && (!weight16 || !weight32)) return FL_ERR_INVALID_ARGUMENT;
  if (!aligned(radius_logit, 4) || !aligned(theta, 4) || !aligned(tr, 4) || !aligned(ti, 4) ||
      !aligned(gamma, 4) || !aligned(weight32, 4) || !aligned(weight16, 2))
    return FL_ERR_INVALID_ARGUMENT;
  const int64_t n = C > n_weight ? C : n_weight;
  fl_field_params_kernel<<<(unsigned)cdiv(n, 256), 256, 0, static_cast<hipStream_t>(stream)>>>(
      radius_logit, theta, (int)C, static_cast<const bf16_bits*>(weight16), (int)n_weight, tr, ti,
      gamma, weight32);
  return hip_status(hipGetLastError());
}

}  // extern "C"
