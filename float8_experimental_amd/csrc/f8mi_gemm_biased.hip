// The forward product of a linear with a bias: the tile kernels with the bias added to the rounded product, the bits of the product and a
// pass that adds the bias, without that pass (4096 x 4096 over 4096, fp32 bias: the product 50.5 us, the bias converted 4.5 and added 15.9;
// with the bias inside 52).  Kernels of their own: the second rounding is eight vector instructions a piece in a last step that the vector
// ALU bounds, which a product without a bias does not pay.  Operands as they are, k-blocked, e4m3 both.
#include "f8mi_gemm_dma16_impl.h"
#include "f8mi_gemm_mid_impl.h"

namespace f8mi {

struct BiasedArgs {
    const uint8_t *A, *Bt;
    int64_t a_unit, b_unit;
    int M, N, K;
    const float *sa, *sb;
    void* C;
    int64_t ldc;
    const void* bias;
    int bias_fp32, tiles_m, tiles_n, c_vec_ok;
};

template <int C_DT, bool ODD, bool ODD_ROWS, int TJ>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_biased_large_kernel(const BiasedArgs g) {
    gemm_dma16_tile<0, 0, C_DT, ODD, false, false, ODD_ROWS, TJ, true>(blockIdx.x, gridDim.x, g.A, 64, g.a_unit, g.Bt, 64, g.b_unit, g.M, g.N, g.K, g.sa, g.sb, g.C,
                                                                       g.ldc, g.bias, g.tiles_m, g.tiles_n, g.c_vec_ok, g.bias_fp32);
}
template <int C_DT, bool ODD_ROWS, int TJ>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_biased_mid_kernel(const BiasedArgs g) {
    gemm_mid_tile<0, 0, C_DT, TJ, false, false, ODD_ROWS, true>(blockIdx.x, gridDim.x, 0, g.A, 64, g.a_unit, g.Bt, 64, g.b_unit, g.M, g.N, g.K, g.sa, g.sb, g.C,
                                                                g.ldc, g.bias, g.tiles_m, g.tiles_n, g.c_vec_ok, 1, g.bias_fp32);
}

template <auto KERNEL, int LDS>
static int launch_biased_kernel(hipStream_t stream, const BiasedArgs& g) {
    static std::atomic<uint64_t> lds_allowed{0};
    if (int rc = allow_big_lds(KERNEL, LDS, lds_allowed)) return rc;
    hipLaunchKernelGGL(KERNEL, dim3((unsigned)(g.tiles_m * g.tiles_n)), dim3(GEMM_THREADS), LDS, stream, g);
    return check_hip(hipGetLastError(), "gemm (with a bias) kernel launch");
}

template <int C_DT, bool ODD_ROWS>
static int launch_biased(bool large, int cols, hipStream_t stream, const BiasedArgs& g) {
    if (!large) {
        if (cols == 128) return launch_biased_kernel<gemm_biased_mid_kernel<C_DT, ODD_ROWS, 4>, MidCfg<4>::LDS>(stream, g);
        return launch_biased_kernel<gemm_biased_mid_kernel<C_DT, ODD_ROWS, 8>, MidCfg<8>::LDS>(stream, g);
    }
    const bool odd = (g.K / 128) & 1;
    if constexpr (!ODD_ROWS) {
        if (cols == 224 && odd) return launch_biased_kernel<gemm_biased_large_kernel<C_DT, true, false, 7>, LargeCfg<7>::LDS>(stream, g);
        if (cols == 224) return launch_biased_kernel<gemm_biased_large_kernel<C_DT, false, false, 7>, LargeCfg<7>::LDS>(stream, g);
    }
    if (odd) return launch_biased_kernel<gemm_biased_large_kernel<C_DT, true, ODD_ROWS, 8>, LargeCfg<8>::LDS>(stream, g);
    return launch_biased_kernel<gemm_biased_large_kernel<C_DT, false, ODD_ROWS, 8>, LargeCfg<8>::LDS>(stream, g);
}

int launch_gemm_biased(bool large, int cols, int c_dtype, hipStream_t stream, const uint8_t* A, int64_t a_unit, const uint8_t* Bt, int64_t b_unit, int M, int N,
                       int K, const float* sa, const float* sb, void* C, int64_t ldc, const void* bias, int bias_fp32, int c_vec_ok) {
    const int rows = large ? 256 : 128;
    const BiasedArgs g{A, Bt, a_unit, b_unit, M, N, K, sa, sb, C, ldc, bias, bias_fp32, (M + rows - 1) / rows, (N + cols - 1) / cols, c_vec_ok};
    const bool odd_rows = c_vec_ok && rows_at_odd_addresses(C, ldc, c_dtype);
    if (c_dtype == F8MI_FP32) return launch_biased<F8MI_FP32, false>(large, cols, stream, g);
    if (c_dtype == F8MI_FP16) return odd_rows ? launch_biased<F8MI_FP16, true>(large, cols, stream, g) : launch_biased<F8MI_FP16, false>(large, cols, stream, g);
    return odd_rows ? launch_biased<F8MI_BF16, true>(large, cols, stream, g) : launch_biased<F8MI_BF16, false>(large, cols, stream, g);
}

}  // namespace f8mi
