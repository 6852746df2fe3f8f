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

// The products |x * scale| up to which the conversion instruction alone gives what clamping first does: it rounds to nearest, so
// everything below the middle between the largest finite code and the next one (464, 61440) becomes that largest code.
template <int FMT>
__device__ __forceinline__ bool within_range(float amax, float scale) {  // amax: of the elements in question; a NaN is outside
    return __builtin_fabsf(__fmul_rn(amax, scale)) <= (FMT == F8MI_E4M3FN ? 460.0f : 60000.0f);
}

// Two adjacent elements within that range -> two fp8 bytes in the lower (HI: upper) half of `old`.  No clamp and no NaN to keep: bf16
// takes three instructions an element (unpack, multiply and half of two conversions) where scale_clamp2 and cvt4_fp8 take seven, which is
// what a cast waits for that has its tile in registers: resident cast of 4096 x 4096 bf16 19.2 -> 17.6 us, 2048 x 4096 12.5 -> 11.5.  Casts of
// larger tensors, which the memory bounds, take what they took.
template <int PROD, int FMT, bool HI>
__device__ __forceinline__ uint32_t cast2_within(float x0, float x1, float scale, uint32_t old) {
    typedef short s2 __attribute__((ext_vector_type(2)));
    const float p0 = __fmul_rn(x0, scale), p1 = __fmul_rn(x1, scale);
    if constexpr (PROD == F8MI_BF16) {
        typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
        const bf2 p = __builtin_bit_cast(bf2, pack_bf16x2(p0, p1));
        const s2 o = __builtin_bit_cast(s2, old);
        if constexpr (FMT == F8MI_E4M3FN) return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(o, p, 1.0f, HI));
        else return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf8_bf16(o, p, 1.0f, HI));
    } else {
        const float q0 = PROD == F8MI_FP16 ? round_to_fp16(p0) : p0, q1 = PROD == F8MI_FP16 ? round_to_fp16(p1) : p1;
        if constexpr (FMT == F8MI_E4M3FN) return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(q0, q1, (int)old, HI);
        else return (uint32_t)__builtin_amdgcn_cvt_pk_bf8_f32(q0, q1, (int)old, HI);
    }
}

// Four elements -> four fp8 bytes in one dword.  WITHIN: within_range holds for their maximum.
template <int PROD, int FMT, bool WITHIN>
__device__ __forceinline__ uint32_t cast4(float x0, float x1, float x2, float x3, float scale) {
    if constexpr (WITHIN) return cast2_within<PROD, FMT, true>(x2, x3, scale, cast2_within<PROD, FMT, false>(x0, x1, scale, 0u));
    constexpr float fmax = FMT == F8MI_E4M3FN ? 448.0f : 57344.0f;
    float f[4];
    scale_clamp2<PROD>(x0, x1, scale, fmax, f[0], f[1]);
    scale_clamp2<PROD>(x2, x3, scale, fmax, f[2], f[3]);
    return cvt4_fp8<FMT>(f[0], f[1], f[2], f[3]);
}

}  // namespace f8mi
