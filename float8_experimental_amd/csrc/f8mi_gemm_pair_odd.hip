// Two products in one launch, operands as they are, 16-bit rows of C at odd multiples of two bytes.
#include "f8mi_gemm_pair_impl.h"

namespace f8mi {

int launch_gemm_pair_odd(bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (c_dtype == F8MI_FP16) {
        if (wide) return launch_pair<F8MI_FP16, F8MI_FP16_IN_FP32, false, true>(stream, pair, second_first);
        return launch_pair<F8MI_FP16, F8MI_FP16, false, true>(stream, pair, second_first);
    }
    if (wide) return launch_pair<F8MI_BF16, F8MI_BF16_IN_FP32, false, true>(stream, pair, second_first);
    return launch_pair<F8MI_BF16, F8MI_BF16, false, true>(stream, pair, second_first);
}

}  // namespace f8mi
