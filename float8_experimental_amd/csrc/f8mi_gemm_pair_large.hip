// Two products in one launch on 256 x 256 tiles, operands as they are.
#include "f8mi_gemm_pair_large_impl.h"

namespace f8mi {

template <int C_DT, int C_WIDE>
static int launch_pair_large_16(bool odd_rows, bool wide, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (odd_rows && wide) return launch_pair_large<C_DT, C_WIDE, false, true>(stream, pair, second_first);
    if (odd_rows) return launch_pair_large<C_DT, C_DT, false, true>(stream, pair, second_first);
    if (wide) return launch_pair_large<C_DT, C_WIDE, false, false>(stream, pair, second_first);
    return launch_pair_large<C_DT, C_DT, false, false>(stream, pair, second_first);
}

int launch_gemm_pair_large(bool transposed, bool odd_rows, bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (transposed) return launch_gemm_pair_large_tr(wide, c_dtype, stream, pair, second_first);
    if (c_dtype == F8MI_FP32) return launch_pair_large<F8MI_FP32, F8MI_FP32, false, false>(stream, pair, second_first);
    if (c_dtype == F8MI_FP16) return launch_pair_large_16<F8MI_FP16, F8MI_FP16_IN_FP32>(odd_rows, wide, stream, pair, second_first);
    return launch_pair_large_16<F8MI_BF16, F8MI_BF16_IN_FP32>(odd_rows, wide, stream, pair, second_first);
}

}  // namespace f8mi
