// Two products in one launch on 128-row tiles.
#include "f8mi_gemm_mid_impl.h"
#include "f8mi_gemm_pair.h"

namespace f8mi {

// C_Q: the type of the second product's C.
template <int C_DT, int C_Q, int TJ, bool TR, bool ODD_ROWS>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_pair_mid_kernel(const GemmPair pair, int second_first) {
    const int bid = blockIdx.x, first = workgroups(pair.s[second_first]);
    const int which = (bid >= first) ^ second_first;
    const int id = bid >= first ? bid - first : bid;
    const GemmSide s = pair.s[which];
    if constexpr (!TR && C_DT == C_Q)
        gemm_mid_tile<1, 0, C_DT, TJ, false, false, ODD_ROWS>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc,
                                                              nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
    else if (which)
        gemm_mid_tile<1, 0, C_Q, TJ, TR, TR, ODD_ROWS && !c_is_fp32(C_Q)>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb,
                                                                         s.C, s.ldc, nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
    else
        gemm_mid_tile<1, 0, C_DT, TJ, false, TR, ODD_ROWS>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc,
                                                           nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
}

template <int C_DT, int C_Q, int TJ, bool TR, bool ODD_ROWS>
static int launch_pair_mid2(hipStream_t stream, const GemmPair& pair, bool second_first) {
    static std::atomic<uint64_t> lds_allowed{0};
    auto kern = gemm_pair_mid_kernel<C_DT, C_Q, TJ, TR, ODD_ROWS>;
    if (int rc = allow_big_lds(kern, MidCfg<TJ>::LDS, lds_allowed)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)(workgroups(pair.s[0]) + workgroups(pair.s[1]))), dim3(GEMM_THREADS), MidCfg<TJ>::LDS, stream, pair, (int)second_first);
    return check_hip(hipGetLastError(), "gemm (two products, 128-row tiles) kernel launch");
}

template <int C_DT, int C_Q, bool TR, bool ODD_ROWS>
static int launch_pair_mid1(int cols, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (cols == 256) return launch_pair_mid2<C_DT, C_Q, 8, TR, ODD_ROWS>(stream, pair, second_first);
    return launch_pair_mid2<C_DT, C_Q, 4, TR, ODD_ROWS>(stream, pair, second_first);
}

template <int C_DT, int C_Q>
static int launch_pair_mid(bool transposed, bool odd_rows, int cols, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (transposed) return launch_pair_mid1<C_DT, C_Q, true, false>(cols, stream, pair, second_first);
    if constexpr (!c_is_fp32(C_DT)) {
        if (odd_rows) return launch_pair_mid1<C_DT, C_Q, false, true>(cols, stream, pair, second_first);
    }
    return launch_pair_mid1<C_DT, C_Q, false, false>(cols, stream, pair, second_first);
}

int launch_gemm_pair_mid(bool transposed, bool odd_rows, bool wide, int cols, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (c_dtype == F8MI_FP32) return launch_pair_mid<F8MI_FP32, F8MI_FP32>(transposed, odd_rows, cols, stream, pair, second_first);
    if (c_dtype == F8MI_FP16) {
        if (wide) return launch_pair_mid<F8MI_FP16, F8MI_FP16_IN_FP32>(transposed, odd_rows, cols, stream, pair, second_first);
        return launch_pair_mid<F8MI_FP16, F8MI_FP16>(transposed, odd_rows, cols, stream, pair, second_first);
    }
    if (wide) return launch_pair_mid<F8MI_BF16, F8MI_BF16_IN_FP32>(transposed, odd_rows, cols, stream, pair, second_first);
    return launch_pair_mid<F8MI_BF16, F8MI_BF16>(transposed, odd_rows, cols, stream, pair, second_first);
}

}  // namespace f8mi
