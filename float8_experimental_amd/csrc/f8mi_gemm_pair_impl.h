// Two products in one launch, each on tiles of its own: 128 x 128, 128 x 256 or 256 x 256.  One kernel holds the bodies of all three (a
// workgroup has a CU to itself on any of them, and the branch is the same for all of its waves), so that any two can be put together.
#pragma once
#include "f8mi_gemm_dma16_impl.h"
#include "f8mi_gemm_mid_impl.h"
#include "f8mi_gemm_pair.h"

namespace f8mi {

constexpr int PAIR_LDS = LargeCfg<8>::LDS > MidCfg<4>::LDS ? LargeCfg<8>::LDS : MidCfg<4>::LDS;
static_assert(PAIR_LDS >= MidCfg<8>::LDS, "the LDS of every body");

template <int C_DT, bool A_TR, bool B_TR, bool ODD_ROWS>
__device__ __forceinline__ void gemm_pair_side(int id, const GemmSide& s) {
    if (s.tiles == F8MI_PAIR_TILES256) {
        if ((s.K / 128) & 1)
            gemm_dma16_tile<1, 0, C_DT, true, A_TR, B_TR, ODD_ROWS, 8>(id, workgroups(s), s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C,
                                                                       s.ldc, nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok);
        else
            gemm_dma16_tile<1, 0, C_DT, false, A_TR, B_TR, ODD_ROWS, 8>(id, workgroups(s), s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C,
                                                                        s.ldc, nullptr, s.tiles_m, s.tiles_n, s.c_vec_ok);
    } else if (s.tiles == F8MI_PAIR_TILES128X256) {
        gemm_mid_tile<1, 0, C_DT, 8, A_TR, B_TR, ODD_ROWS>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc, nullptr,
                                                           s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
    } else {
        gemm_mid_tile<1, 0, C_DT, 4, A_TR, B_TR, ODD_ROWS>(id, workgroups(s), 0, s.A, s.lda, s.a_unit, s.Bt, s.ldb, s.b_unit, s.M, s.N, s.K, s.sa, s.sb, s.C, s.ldc, nullptr,
                                                           s.tiles_m, s.tiles_n, s.c_vec_ok, 1);
    }
}

// C_Q: the type of the second product's C.
template <int C_DT, int C_Q, bool TR, bool ODD_ROWS>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_pair_kernel(const GemmPair pair, int second_first) {
    const int bid = blockIdx.x, first = workgroups(pair.s[second_first]);
    const int which = (bid >= first) ^ second_first;
    const int id = bid >= first ? bid - first : bid;
    const GemmSide s = pair.s[which];
    if constexpr (!TR && C_DT == C_Q) gemm_pair_side<C_DT, false, false, ODD_ROWS>(id, s);
    else if (which) gemm_pair_side<C_Q, TR, TR, ODD_ROWS && !c_is_fp32(C_Q)>(id, s);
    else gemm_pair_side<C_DT, false, TR, ODD_ROWS>(id, s);
}

template <int C_DT, int C_Q, bool TR, bool ODD_ROWS>
static int launch_pair(hipStream_t stream, const GemmPair& pair, bool second_first) {
    static std::atomic<uint64_t> lds_allowed{0};
    auto kern = gemm_pair_kernel<C_DT, C_Q, TR, ODD_ROWS>;
    if (int rc = allow_big_lds(kern, PAIR_LDS, lds_allowed)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)(workgroups(pair.s[0]) + workgroups(pair.s[1]))), dim3(GEMM_THREADS), PAIR_LDS, stream, pair, (int)second_first);
    return check_hip(hipGetLastError(), "gemm (two products) kernel launch");
}

}  // namespace f8mi
