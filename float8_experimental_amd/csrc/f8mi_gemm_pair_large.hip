// Two products in one launch on 256 x 256 tiles, operands as they are.
#include "f8mi_gemm_pair_large_impl.h"

namespace f8mi {

int launch_gemm_pair_large(bool transposed, bool odd_rows, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (transposed) return launch_gemm_pair_large_tr(c_dtype, stream, pair, second_first);
    if (c_dtype == F8MI_FP32) return launch_pair_large<F8MI_FP32, false, false>(stream, pair, second_first);
    if (c_dtype == F8MI_FP16) {
        if (odd_rows) return launch_pair_large<F8MI_FP16, false, true>(stream, pair, second_first);
        return launch_pair_large<F8MI_FP16, false, false>(stream, pair, second_first);
    }
    if (odd_rows) return launch_pair_large<F8MI_BF16, false, true>(stream, pair, second_first);
    return launch_pair_large<F8MI_BF16, false, false>(stream, pair, second_first);
}

}  // namespace f8mi
