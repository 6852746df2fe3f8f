// The arithmetic of the saturated cast, shared by the kernels that write fp8 tensors and those that convert in registers.
#pragma once
#include "f8mi_common.h"

namespace f8mi {

// clamp to [-fmax, fmax], NaN kept (v_med3_f32 drops it, so it is put back)
__device__ __forceinline__ float clamp_keep_nan(float y, float fmax) {
    const float c = __builtin_amdgcn_fmed3f(y, -fmax, fmax);
    return (y != y) ? y : c;
}

// Two adjacent elements: x*scale rounded to PROD, clamped, as fp32 ready for conversion.
template <int PROD>
__device__ __forceinline__ void scale_clamp2(float x0, float x1, float scale, float fmax, float& y0, float& y1) {
    float p0 = __fmul_rn(x0, scale), p1 = __fmul_rn(x1, scale);
    if constexpr (PROD == F8MI_BF16) {
        const uint32_t w = pack_bf16x2(p0, p1);
        p0 = __uint_as_float(w << 16);
        p1 = __uint_as_float(w & 0xffff0000u);
    } else if constexpr (PROD == F8MI_FP16) {
        p0 = round_to_fp16(p0);
        p1 = round_to_fp16(p1);
    }
    y0 = clamp_keep_nan(p0, fmax);
    y1 = clamp_keep_nan(p1, fmax);
}

}  // namespace f8mi
