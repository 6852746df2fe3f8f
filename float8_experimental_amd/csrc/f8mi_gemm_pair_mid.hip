// Two products in one launch on 128-row tiles.
#include "f8mi_gemm_mid_impl.h"
#include "f8mi_gemm_pair.h"

namespace f8mi {

template <int C_DT, int TJ, bool TR, bool ODD_ROWS>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_pair_mid_kernel(const GemmPair pair, int second_first) {
    const int bid = blockIdx.x, first = workgroups(pair.s[second_first]);
    const int which = (bid >= first) ^ second_first;
    const int id = bid >= first ? bid - first : bid;
    const GemmSide s = pair.s[which];
    if constexpr (!TR)
        gemm_mid_tile<1, 0, C_DT, TJ, false, false, ODD_ROWS>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc,
                                                                 nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
    else if (which)
        gemm_mid_tile<1, 0, C_DT, TJ, true, true, ODD_ROWS>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc,
                                                               nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
    else
        gemm_mid_tile<1, 0, C_DT, TJ, false, true, ODD_ROWS>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc,
                                                                nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
}

template <int C_DT, int TJ, bool TR, bool ODD_ROWS>
static int launch_pair_mid2(hipStream_t stream, const GemmPair& pair, bool second_first) {
    static std::atomic<uint64_t> lds_allowed{0};
    auto kern = gemm_pair_mid_kernel<C_DT, TJ, TR, ODD_ROWS>;
    if (int rc = allow_big_lds(kern, MidCfg<TJ>::LDS, lds_allowed)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)(workgroups(pair.s[0]) + workgroups(pair.s[1]))), dim3(GEMM_THREADS), MidCfg<TJ>::LDS, stream, pair, (int)second_first);
    return check_hip(hipGetLastError(), "gemm (two products, 128-row tiles) kernel launch");
}

template <int C_DT, bool TR, bool ODD_ROWS>
static int launch_pair_mid1(bool wide, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (wide) return launch_pair_mid2<C_DT, 8, TR, ODD_ROWS>(stream, pair, second_first);
    return launch_pair_mid2<C_DT, 4, TR, ODD_ROWS>(stream, pair, second_first);
}

int launch_gemm_pair_mid(bool transposed, bool odd_rows, bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (c_dtype == F8MI_FP32)
        return transposed ? launch_pair_mid1<F8MI_FP32, true, false>(wide, stream, pair, second_first) : launch_pair_mid1<F8MI_FP32, false, false>(wide, stream, pair, second_first);
    if (c_dtype == F8MI_FP16) {
        if (transposed) return launch_pair_mid1<F8MI_FP16, true, false>(wide, stream, pair, second_first);
        if (odd_rows) return launch_pair_mid1<F8MI_FP16, false, true>(wide, stream, pair, second_first);
        return launch_pair_mid1<F8MI_FP16, false, false>(wide, stream, pair, second_first);
    }
    if (transposed) return launch_pair_mid1<F8MI_BF16, true, false>(wide, stream, pair, second_first);
    if (odd_rows) return launch_pair_mid1<F8MI_BF16, false, true>(wide, stream, pair, second_first);
    return launch_pair_mid1<F8MI_BF16, false, false>(wide, stream, pair, second_first);
}

}  // namespace f8mi
