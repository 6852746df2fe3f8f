// Two products in one launch, the second one's 16-bit result in fp32.
#include "f8mi_gemm_pair_impl.h"

namespace f8mi {

int launch_gemm_pair_wide(bool transposed, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first) {
    if (c_dtype == F8MI_FP16) {
        if (transposed) return launch_pair<F8MI_FP16, F8MI_FP16_IN_FP32, true, false>(stream, pair, second_first);
        return launch_pair<F8MI_FP16, F8MI_FP16_IN_FP32, false, false>(stream, pair, second_first);
    }
    if (transposed) return launch_pair<F8MI_BF16, F8MI_BF16_IN_FP32, true, false>(stream, pair, second_first);
    return launch_pair<F8MI_BF16, F8MI_BF16_IN_FP32, false, false>(stream, pair, second_first);
}

}  // namespace f8mi
