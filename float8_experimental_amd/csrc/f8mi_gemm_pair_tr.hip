// Two products in one launch: Bt of one read transposed, both operands of the other.
#include "f8mi_gemm_pair_impl.h"

namespace f8mi {

int launch_gemm_pair_tr(bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (wide) return launch_gemm_pair_wide(true, c_dtype, stream, pair, second_first);
    if (c_dtype == F8MI_FP32) return launch_pair<F8MI_FP32, F8MI_FP32, true, false>(stream, pair, second_first);
    if (c_dtype == F8MI_FP16) return launch_pair<F8MI_FP16, F8MI_FP16, true, false>(stream, pair, second_first);
    return launch_pair<F8MI_BF16, F8MI_BF16, true, false>(stream, pair, second_first);
}

}  // namespace f8mi
