// Two products in one launch (the backward of a linear: grad_input and grad_weight): what the host rule and the kernels share.
//
// One after the other, each product fills the chip and drains it again, and the workgroups of its last round leave the rest of the CUs idle.
// In one launch the tiles of the second start where those of the first end, those of the longer contraction first.  Both products have the
// same work, so a product of few tiles that each take long runs beside one of many that do not.  us back to back, one after the other / together (tokens,
// in -> out features; tiles): 512, 1024 -> 1024: 12.4 / 7.2 (128 x 128); 384, 2048 -> 5120: 28.4 / 18.7 (128 x 128 and 256 x 256); 1664, 3328 -> 2560:
// 41.0 / 30.1 (256 x 256); 2048, 4096 -> 4096: 55.8 / 51.8 (256 x 256); 3584, 2816 -> 11648: 187 / 164; 2981, 2989 -> 8117: 141 / 117; where the rule in
// f8mi_gemm.hip stays with two: 4096, 4096 -> 4096, one full round each: 93.7 / 94.1; 8192, 4096 -> 14336: 616 / 619.  Tiles of the
// first and of the second product, the best two of one kind / of their own as chosen: 7040, 2560 -> 512: 32.4 / 28.8; 8192, 4096 -> 1024: 66.4 / 62.7; 1209, 1408 ->
// 6144: 29.5 / 23.5.  Few tokens in wide layers gain little: 512, 6400 -> 15232: 150 / 149, though 135 with 128 x 128 beside 256 x 256, which the estimate does not see.
// The tiles are the ones that a product by itself runs on (f8mi_gemm_dma16_impl.h, f8mi_gemm_mid_impl.h): the same bits.
#pragma once
#include "f8mi_gemm_util.h"

namespace f8mi {

// One product: the arguments of its kernel by itself.
struct GemmSide {
    const uint8_t* A;
    int64_t lda, a_unit;
    const uint8_t* Bt;
    int64_t ldb, b_unit;
    int M, N, K;
    const float *sa, *sb;
    void* C;
    int64_t ldc;
    int tiles_m, tiles_n;
    int c_vec_ok;
    int tiles;  // F8MI_PAIR_TILES128, _TILES128X256 or _TILES256
};

__host__ __device__ inline int workgroups(const GemmSide& s) { return s.tiles_m * s.tiles_n; }
// Both, as a kernel takes them: the side is looked up by its index, one set of scalar registers for either (as two arguments their fields
// are all loaded up front, and 90 scalar registers spilled).
struct GemmPair {
    GemmSide s[2];
};
// A e5m2, Bt e4m3 on both sides.  transposed: s[0] reads its Bt transposed, s[1] both its operands; else both sides read them as they are.
// second_first: the workgroups of s[1] come first.
// odd_rows: rows of C at odd multiples of two bytes (not with transposed; of s[0] only where s[1] is wide).
// wide: C of s[1] is fp32 that holds values of c_dtype (bf16, fp16).
int launch_gemm_pair(bool transposed, bool odd_rows, bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first);
int launch_gemm_pair_tr(bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first);
int launch_gemm_pair_odd(bool wide, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first);
int launch_gemm_pair_wide(bool transposed, int c_dtype, hipStream_t stream, const GemmPair& pair, bool second_first);
// One product with such a C (f8mi_gemm_wide.hip): e5m2 times e4m3, both operands as they are or both transposed; large: tiles of 256 x cols
// (256, or, operands as they are, 224), else 128 x cols (128, 256).
int launch_gemm_wide(bool transposed, bool large, int cols, int c_dtype, hipStream_t stream, const GemmSide& s);

}  // namespace f8mi
