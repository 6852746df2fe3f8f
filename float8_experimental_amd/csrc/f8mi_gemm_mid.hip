// The 128-row-tile GEMM on operands as they are, and its split over k.
#include "f8mi_gemm_mid_impl.h"

namespace f8mi {

// wide: 128 x 256 tiles instead of 128 x 128
int launch_gemm_mid(int a_fmt, int b_fmt, int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                    const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                    int64_t ldc, const void* bias, int c_vec_ok) {
    if (c_vec_ok && rows_at_odd_addresses(C, ldc, c_dtype))
        return launch_gemm_mid_odd(a_fmt, b_fmt, c_dtype, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok);
    return launch_mid1<false, false>(a_fmt, b_fmt, c_dtype, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, 1);
}

// C = (partial[0] + partial[1] + ... in this order) / (sa * sb) + bias: four neighbouring columns per lane (N % 4 == 0)
template <int C_DT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ partial, int k_splits, int M, int N,
                                                            const float* __restrict__ sa_dev, const float* __restrict__ sb_dev,
                                                            void* __restrict__ C, int64_t ldc, const void* __restrict__ bias, int c_vec_ok) {
    const int64_t quads = (int64_t)N / 4;
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= (int64_t)M * quads) return;
    const int64_t row = q / quads;
    const int col = (int)(q % quads) * 4;
    const float inv = __fdiv_rn(1.0f, *sa_dev) * __fdiv_rn(1.0f, *sb_dev);
    const int64_t slab = (int64_t)M * N;
    float4 sum = *(const float4*)(partial + row * N + col);
    for (int s = 1; s < k_splits; s++) {
        const float4 p = *(const float4*)(partial + s * slab + row * N + col);
        sum.x += p.x; sum.y += p.y; sum.z += p.z; sum.w += p.w;
    }
    float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = v[e] * inv + (bias ? load_bias<C_DT>(bias, col + e) : 0.f);
    if constexpr (C_DT == F8MI_FP32) {
        float* dst = (float*)C + row * ldc + col;
        if (c_vec_ok) {
            store16_any(dst, make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])));
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) dst[e] = v[e];
        }
    } else {
        uint16_t* dst = (uint16_t*)C + row * ldc + col;
        const uint32_t p0 = pack2<C_DT>(v[0], v[1]), p1 = pack2<C_DT>(v[2], v[3]);
        if (c_vec_ok) {  // one 8-byte store at element alignment
            store8_any(dst, p0, p1);
        } else {
            dst[0] = (uint16_t)(p0 & 0xffffu); dst[1] = (uint16_t)(p0 >> 16);
            dst[2] = (uint16_t)(p1 & 0xffffu); dst[3] = (uint16_t)(p1 >> 16);
        }
    }
}

// The contraction split k_splits ways over workgroups (outputs of few tiles and a long k: every CU gets a part).
// `partial` holds k_splits x M x N floats (16-byte aligned); host side has checked K % (128 * k_splits) == 0, N % 4 == 0.
int launch_gemm_mid_splitk(int a_fmt, int b_fmt, int c_dtype, bool wide, int k_splits, float* partial, hipStream_t stream, const uint8_t* A,
                           int64_t lda, int64_t a_unit, const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa,
                           const float* sb, void* C, int64_t ldc, const void* bias, int c_vec_ok) {
    if (int rc = launch_mid1<false, false>(a_fmt, b_fmt, F8MI_FP32, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, partial, N, nullptr, 1, k_splits))
        return rc;
    const int64_t quads = (int64_t)M * (N / 4);
    const dim3 grid((unsigned)((quads + 255) / 256));
    if (c_dtype == F8MI_BF16) hipLaunchKernelGGL(splitk_reduce_kernel<F8MI_BF16>, grid, dim3(256), 0, stream, partial, k_splits, M, N, sa, sb, C, ldc, bias, c_vec_ok);
    else if (c_dtype == F8MI_FP16) hipLaunchKernelGGL(splitk_reduce_kernel<F8MI_FP16>, grid, dim3(256), 0, stream, partial, k_splits, M, N, sa, sb, C, ldc, bias, c_vec_ok);
    else hipLaunchKernelGGL(splitk_reduce_kernel<F8MI_FP32>, grid, dim3(256), 0, stream, partial, k_splits, M, N, sa, sb, C, ldc, bias, c_vec_ok);
    return check_hip(hipGetLastError(), "gemm split-k reduction kernel launch");
}

}  // namespace f8mi
