// The 128-row-tile GEMM for 2-byte outputs with rows at odd multiples of two bytes.
#include "f8mi_gemm_mid_impl.h"

namespace f8mi {

int launch_gemm_mid_odd(int a_fmt, int b_fmt, int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                        const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                        int64_t ldc, const void* bias, int c_vec_ok) {
    return launch_mid1<false, false, true>(a_fmt, b_fmt, c_dtype, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, 1);
}

}  // namespace f8mi
