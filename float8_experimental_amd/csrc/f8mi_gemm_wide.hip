// A product whose 16-bit result is stored in fp32: the gradient of an fp32 weight under autocast, without the pass that converts it (4096 x 4096
// over 4096, both operands transposed: the product 49 us and torch's conversion 17; stored in fp32 53).  The tile kernels of
// f8mi_gemm_dma16_impl.h and f8mi_gemm_mid_impl.h, e5m2 times e4m3, both operands as they are or both read transposed.
#include "f8mi_gemm_dma16_impl.h"
#include "f8mi_gemm_mid_impl.h"
#include "f8mi_gemm_pair.h"

namespace f8mi {

template <int C_DT, bool TR, bool ODD, int TJ>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_wide_large_kernel(const GemmSide s) {
    gemm_dma16_tile<1, 0, C_DT, ODD, TR, TR, false, TJ>(blockIdx.x, gridDim.x, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc, nullptr,
                                                        s.tiles_m, s.tiles_n, s.c_vec_ok);
}
template <int C_DT, bool TR, int TJ>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_wide_mid_kernel(const GemmSide s) {
    gemm_mid_tile<1, 0, C_DT, TJ, TR, TR, false>(blockIdx.x, gridDim.x, 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc, nullptr,
                                                 s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
}

template <auto KERNEL, int LDS>
static int launch_wide_kernel(hipStream_t stream, const GemmSide& s) {
    static std::atomic<uint64_t> lds_allowed{0};
    if (int rc = allow_big_lds(KERNEL, LDS, lds_allowed)) return rc;
    hipLaunchKernelGGL(KERNEL, dim3((unsigned)workgroups(s)), dim3(GEMM_THREADS), LDS, stream, s);
    return check_hip(hipGetLastError(), "gemm (16-bit result in fp32) kernel launch");
}

template <int C_DT, bool TR>
static int launch_wide(bool large, int cols, hipStream_t stream, const GemmSide& s) {
    if (!large) {
        if (cols == 128) return launch_wide_kernel<gemm_wide_mid_kernel<C_DT, TR, 4>, MidCfg<4>::LDS>(stream, s);
        return launch_wide_kernel<gemm_wide_mid_kernel<C_DT, TR, 8>, MidCfg<8>::LDS>(stream, s);
    }
    const bool odd = (s.K / 128) & 1;
    if constexpr (!TR) {
        if (cols == 224 && odd) return launch_wide_kernel<gemm_wide_large_kernel<C_DT, false, true, 7>, LargeCfg<7>::LDS>(stream, s);
        if (cols == 224) return launch_wide_kernel<gemm_wide_large_kernel<C_DT, false, false, 7>, LargeCfg<7>::LDS>(stream, s);
    }
    if (odd) return launch_wide_kernel<gemm_wide_large_kernel<C_DT, TR, true, 8>, LargeCfg<8>::LDS>(stream, s);
    return launch_wide_kernel<gemm_wide_large_kernel<C_DT, TR, false, 8>, LargeCfg<8>::LDS>(stream, s);
}

int launch_gemm_wide(bool transposed, bool large, int cols, int c_dtype, hipStream_t stream, const GemmSide& side) {
    GemmSide s = side;
    const int rows = large ? 256 : 128;
    s.tiles_m = (s.M + rows - 1) / rows;
    s.tiles_n = (s.N + cols - 1) / cols;
    if (c_dtype == F8MI_FP16_IN_FP32) return transposed ? launch_wide<F8MI_FP16_IN_FP32, true>(large, cols, stream, s) : launch_wide<F8MI_FP16_IN_FP32, false>(large, cols, stream, s);
    return transposed ? launch_wide<F8MI_BF16_IN_FP32, true>(large, cols, stream, s) : launch_wide<F8MI_BF16_IN_FP32, false>(large, cols, stream, s);
}

}  // namespace f8mi
