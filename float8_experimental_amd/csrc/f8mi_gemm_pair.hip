// Two products in one launch, operands as they are, results of one type.
#include "f8mi_gemm_pair_impl.h"

namespace f8mi {

int launch_gemm_pair(bool transposed, bool odd_rows, bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (transposed) return launch_gemm_pair_tr(wide, c_dtype, stream, pair, second_first);
    if (odd_rows) return launch_gemm_pair_odd(wide, c_dtype, stream, pair, second_first);
    if (wide) return launch_gemm_pair_wide(false, c_dtype, stream, pair, second_first);
    if (c_dtype == F8MI_FP32) return launch_pair<F8MI_FP32, F8MI_FP32, false, false>(stream, pair, second_first);
    if (c_dtype == F8MI_FP16) return launch_pair<F8MI_FP16, F8MI_FP16, false, false>(stream, pair, second_first);
    return launch_pair<F8MI_BF16, F8MI_BF16, false, false>(stream, pair, second_first);
}

}  // namespace f8mi
