// Pieces shared by the two fp8 GEMM kernels (register-staged and LDS-DMA): tile constants,
// fragment reads, output conversion and the C epilogue.
#pragma once
#include <atomic>
#include <type_traits>

#include "f8mi_common.h"

namespace f8mi {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int BM = 256, BN = 256, BK = 128;
constexpr int GEMM_THREADS = 256;
constexpr int STAGE_BYTES = (BM + BN) * BK;  // 64 KB
constexpr int EPI_PITCH = 128 * 2 + 16;      // bytes per row of a wave's 128 x 128 2-byte output tile in LDS
constexpr int EPI_BYTES = 4 * 128 * EPI_PITCH;
constexpr int GEMM_LDS = 2 * STAGE_BYTES > EPI_BYTES ? 2 * STAGE_BYTES : EPI_BYTES;
constexpr int GROUP_M = 8;
constexpr int NUM_XCD = 8;

// Consecutive workgroup ids go to the 8 XCDs round-robin.  Re-deals them so that XCD x (ids x, x+8, ...) works on
// a contiguous run of the tile order -- whatever the grid size: the first `grid % 8` XCDs get one workgroup more.
__device__ __forceinline__ int xcd_contiguous_id(int bid, int grid) {
    const int x = bid % NUM_XCD, q = grid / NUM_XCD, r = grid % NUM_XCD;
    return x * q + min(x, r) + bid / NUM_XCD;
}

#define F8MI_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

__device__ __forceinline__ v8i read_frag(const uint8_t* p0, const uint8_t* p1) {
    const uint4 lo = *(const uint4*)p0;
    const uint4 hi = *(const uint4*)p1;
    return (v8i){(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}

typedef int v2i __attribute__((ext_vector_type(2)));

// Four transpose reads = the 32 contraction bytes of one lane's MFMA operand (rows k0 + 8t .. + 7, t = 0..3, of
// the lane's column): in every group of 16 lanes, lane i receives byte i%8 of the 8 bytes addressed by lanes
// 2b + i/8 (b = 0..7); callers point lane j at (row k0 + j/2, column n0 + 8*(j%2)), so lane i gets column n0 + i.
template <int ROW_BYTES = 256>
__device__ __forceinline__ v8i read_frag_tr(const uint8_t* p) {
    typedef __attribute__((address_space(3))) v2i* lds_v2i;
    const v2i r0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(p));
    const v2i r1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(p + 8 * ROW_BYTES));
    const v2i r2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(p + 16 * ROW_BYTES));
    const v2i r3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i)(p + 24 * ROW_BYTES));
    return (v8i){r0.x, r0.y, r1.x, r1.y, r2.x, r2.y, r3.x, r3.y};
}

// f(k) of the transposed-slab swizzle: the 16-byte slot c of contraction row k sits at slot c ^ f(k).  One
// transpose read touches rows 8t..8t+7 of two 32-row quarters per 32 lanes; f makes those 16 rows hit 16
// different slots.
__device__ __forceinline__ int tr_swizzle(int k) { return (k & 7) | (((k >> 5) & 1) << 3); }

// Types of C: F8MI_BF16, F8MI_FP16, F8MI_FP32, and fp32 that holds the 16-bit result (include/f8mi.h).
constexpr __host__ __device__ bool c_is_fp32(int c_dtype) { return c_dtype >= F8MI_FP32; }
constexpr __host__ __device__ int c_rounded_to(int c_dtype) {
    return c_dtype == F8MI_BF16_IN_FP32 ? F8MI_BF16 : c_dtype == F8MI_FP16_IN_FP32 ? F8MI_FP16 : c_dtype;
}

template <int C_DT>
__device__ __forceinline__ float load_bias(const void* bias, int col) {
    if constexpr (C_DT == F8MI_BF16) return bf16_bits_to_float(((const uint16_t*)bias)[col]);
    else if constexpr (C_DT == F8MI_FP16) return fp16_bits_to_float(((const uint16_t*)bias)[col]);
    else return ((const float*)bias)[col];
}

// The bias of the columns col0 + 16 tj + e, zeros without one; columns past the end get the last one's, which nobody stores.  One
// branch in all: with a test for each element the last step of a 128 x 256 tile began with 64 of them, bias or none (2048 tokens, 4096 -> 14336 with a
// bias: 96.9 -> 93.5 us; a training step of 2048, 4096 -> 4096: 132 -> 131, of 8192, 4096 -> 14336 twice: 2333 -> 2315).
template <int C_DT, int TJ>
__device__ __forceinline__ void load_bias_tiles(float (&bv)[TJ][4], const void* bias, int col0, int N) {
    if (bias) {
#pragma unroll
        for (int tj = 0; tj < TJ; tj++)
#pragma unroll
            for (int e = 0; e < 4; e++) bv[tj][e] = load_bias<C_DT>(bias, min(col0 + 16 * tj + e, N - 1));
    } else {
#pragma unroll
        for (int tj = 0; tj < TJ; tj++)
#pragma unroll
            for (int e = 0; e < 4; e++) bv[tj][e] = 0.f;
    }
}

// two fp32 -> two packed 2-byte outputs (round to nearest even)
template <int C_DT>
__device__ __forceinline__ uint32_t pack2(float a, float b) {
    if constexpr (C_DT == F8MI_BF16) {
        typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
        typedef float f2 __attribute__((ext_vector_type(2)));
        bf2 r = __builtin_convertvector((f2){a, b}, bf2);
        return __builtin_bit_cast(uint32_t, r);
    } else {
        return (uint32_t)__half_as_ushort(__float2half_rn(a)) | ((uint32_t)__half_as_ushort(__float2half_rn(b)) << 16);
    }
}

template <int C_DT>
__device__ __forceinline__ void unpack2(uint32_t w, float& a, float& b) {
    if constexpr (C_DT == F8MI_BF16) {
        a = __uint_as_float(w << 16);
        b = __uint_as_float(w & 0xffff0000u);
    } else {
        a = fp16_bits_to_float(w & 0xffffu);
        b = fp16_bits_to_float(w >> 16);
    }
}

// Two accumulators to two packed 2-byte outputs.  BIAS_AFTER: the product is rounded to the output's type, then the bias (of that type) is
// added and the sum rounded again, as `x @ w.t() + bias` does; else the bias is added before the only rounding.
template <int C_DT, bool BIAS_AFTER>
__device__ __forceinline__ uint32_t finish2(float a, float b, float inv, float bias_a, float bias_b) {
    if constexpr (!BIAS_AFTER) {
        return pack2<C_DT>(a * inv + bias_a, b * inv + bias_b);
    } else {
        float x, y;
        unpack2<C_DT>(pack2<C_DT>(a * inv + 0.f, b * inv + 0.f), x, y);  // + 0: a product of -0 is 0, as without a bias
        return pack2<C_DT>(x + bias_a, y + bias_b);
    }
}
// Four neighbouring columns of an fp32 C.
template <int C_DT, bool BIAS_AFTER>
__device__ __forceinline__ uint4 finish4(const float (&a)[4], float inv, const float (&bias)[4]) {
    constexpr int R = c_rounded_to(C_DT);
    float v[4];
    if constexpr (R != F8MI_FP32) {
        unpack2<R>(pack2<R>(a[0] * inv + bias[0], a[1] * inv + bias[1]), v[0], v[1]);
        unpack2<R>(pack2<R>(a[2] * inv + bias[2], a[3] * inv + bias[3]), v[2], v[3]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = BIAS_AFTER ? __fadd_rn(__fmaf_rn(a[i], inv, 0.f), bias[i]) : a[i] * inv + bias[i];
    }
    return make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3]));
}
// ... and their store, at dst = C[row][col].  whole: all four lie inside C and it takes 16-byte stores (the same for every lane).
__device__ __forceinline__ void store_fp32x4(float* dst, uint4 v, bool whole, int c_vec_ok, int row, int col, int M, int N) {
    if (__builtin_expect(whole, 1)) {
        store16_any(dst, v);
    } else if (row < M && col < N) {
        if (c_vec_ok && col + 4 <= N) {
            store16_any(dst, v);
        } else {
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (col + i < N) ((uint32_t*)dst)[i] = w[i];
        }
    }
}

// load_bias_tiles for BIAS_AFTER: a bias of C's type, or an fp32 one rounded to it.
template <int C_DT, int TJ>
__device__ __forceinline__ void load_rounded_bias_tiles(float (&bv)[TJ][4], const void* bias, int bias_fp32, int col0, int N) {
    if (C_DT == F8MI_FP32 || !bias_fp32) {
        load_bias_tiles<C_DT, TJ>(bv, bias, col0, N);
        return;
    }
    load_bias_tiles<F8MI_FP32, TJ>(bv, bias, col0, N);
    if constexpr (C_DT != F8MI_FP32) {
#pragma unroll
        for (int tj = 0; tj < TJ; tj++)
#pragma unroll
            for (int e = 0; e < 4; e += 2) unpack2<C_DT>(pack2<C_DT>(bv[tj][e], bv[tj][e + 1]), bv[tj][e], bv[tj][e + 1]);
    }
}

// Stores of 2-byte outputs whose rows do not all start at a multiple of four bytes (an odd row pitch): the memory system takes a 16-byte
// store apart unless it starts at one (4096 rows, 11007 columns over 4224: 151 us at pitches 11008, 11006 and 11004, 178 at 11007, now 157;
// 2048 x 4095 over 4096 in 128-row tiles: 33 at an even pitch, 36 at this one).  A lane of such a row stores one column further to the left instead, its neighbour's last column and its own first seven.
// In kernels of their own (ODD_ROWS, operands as they are): inside the others, not even taken, the code cost products of 2048 x 4096 x
// 4096 between other kernels 2 us each.
// Lanes hold 8 neighbouring columns of one row, the quarters lane / 16 = 0, 2, 1, 3 of a wave 32 of them one behind the other; the
// pieces of 32 columns of one row are stored from left to right.
inline bool rows_at_odd_addresses(const void* C, int64_t ldc, int c_dtype) { return !c_is_fp32(c_dtype) && ((ldc & 1) || ((uintptr_t)C & 2)); }
struct ShiftedRows {
    int shifted;      // 1: this lane's rows (16 apart) need it
    uint32_t sel;     // bytes of {a word, the one before it} that make a stored word
    int from;         // ds_bpermute address of the lane that holds the 8 columns before
    uint4 held;       // the piece to be stored next
    uint32_t prev;    // the last word before it

    __device__ __forceinline__ ShiftedRows(const void* C, int64_t ldc, int row) {
        const int lane = threadIdx.x & 63, lq = lane >> 4;
        shifted = (((uintptr_t)C >> 1) + (uint64_t)row * (uint64_t)ldc) & 1;
        sel = shifted ? 0x05040302u : 0x07060504u;
        from = 4 * (lane + (lq == 0 ? 48 : lq == 1 ? 16 : -32));
        held = make_uint4(0u, 0u, 0u, 0u);
        prev = 0u;
    }
    // The lane's columns col .. + 7 of `row`, at dst, in two halves so that the exchange between lanes has the time of the next piece:
    // `hold` takes them, `store` writes what is held.  Every lane takes part.  whole: row and columns lie inside C in every lane.
    __device__ __forceinline__ void hold(uint4 w) {
        const int lq = (threadIdx.x & 63) >> 4;
        prev = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(lq == 3 ? held.w : w.w));
        held = w;
    }
    __device__ __forceinline__ void store(uint16_t* dst, bool whole, bool first, bool last, int row, int col, int M, int N) const {
        const int lq = (threadIdx.x & 63) >> 4;
        const uint32_t d0 = __builtin_amdgcn_perm(held.x, prev, sel), d1 = __builtin_amdgcn_perm(held.y, held.x, sel);
        const uint32_t d2 = __builtin_amdgcn_perm(held.z, held.y, sel), d3 = __builtin_amdgcn_perm(held.w, held.z, sel);
        const bool no_left = first && lq == 0 && shifted;  // the column before belongs to another wave
        if (!whole && (row >= M || col >= N)) return;
        if (!no_left && (whole || col + 8 - shifted <= N)) {
            store16_any(dst - shifted, make_uint4(d0, d1, d2, d3));
        } else if (no_left && (whole || col + 7 <= N)) {
            dst[0] = (uint16_t)held.x;
            store8_any(dst + 1, d1, d2);
            *(u32_any*)(dst + 5) = d3;
        } else {
            const uint32_t v[4] = {held.x, held.y, held.z, held.w};
#pragma unroll
            for (int i = 0; i < 8; i++)
                if (col + i < N) dst[i] = (uint16_t)(v[i >> 1] >> (16 * (i & 1)));
            if (shifted && !no_left) dst[-1] = (uint16_t)d0;
            return;
        }
        // nobody to the right takes the last column
        if (shifted && ((last && lq == 3) || (!whole && col + 8 == N)) && (whole || col + 8 <= N)) dst[7] = (uint16_t)(held.w >> 16);
    }
};

// Scales a workgroup's 256 x 256 accumulators by 1 / (sa * sb), adds the bias, converts and writes C.
// acc[tj][ti] is the 32 x 32 tile (row block ti, column block tj) of this wave's 128 x 128 quarter
// as left by MFMA(first = Bt rows, second = A rows): lane holds row lane%32 and columns
// 8*(e/4) + 4*(lane/32) + e%4.  2-byte outputs go through a padded LDS tile per wave so that C is
// written with 16-byte stores; `smem` must be free for that (EPI_BYTES) when every wave arrives.
template <int C_DT>
__device__ __forceinline__ void store_c_tile(v16f (&acc)[4][4], uint8_t* smem, int m0, int n0, int M, int N,
                                             const float* __restrict__ sa_dev, const float* __restrict__ sb_dev,
                                             void* __restrict__ C, int64_t ldc, const void* __restrict__ bias,
                                             int c_vec_ok) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const float inv = __fdiv_rn(1.0f, *sa_dev) * __fdiv_rn(1.0f, *sb_dev);
    const int lm = lane & 31, lh = lane >> 5;
    const int wrow0 = m0 + wm * 128, wcol0 = n0 + wn * 128;

    if constexpr (C_DT == F8MI_FP32) {
        // 4 consecutive columns per lane = one 16-byte store
        float* Cf = (float*)C;
#pragma unroll
        for (int ti = 0; ti < 4; ti++) {
            const int row = wrow0 + ti * 32 + lm;
#pragma unroll
            for (int tj = 0; tj < 4; tj++) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const int col = wcol0 + tj * 32 + 8 * g + 4 * lh;
                    if (row >= M || col >= N) continue;
                    float v[4];
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        v[r] = acc[tj][ti][4 * g + r] * inv;
                        if (bias && col + r < N) v[r] += load_bias<C_DT>(bias, col + r);
                    }
                    float* dst = Cf + (int64_t)row * ldc + col;
                    if (c_vec_ok && col + 4 <= N) {
                        store16_any(dst, make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])));
                    } else {
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            if (col + r < N) dst[r] = v[r];
                    }
                }
            }
        }
    } else {
        // all waves are done with the operand stages before they become the output staging area
        lds_barrier();
        uint8_t* ep = smem + wave * (128 * EPI_PITCH);
#pragma unroll
        for (int tj = 0; tj < 4; tj++) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const int cl = tj * 32 + 8 * g + 4 * lh;  // column inside the wave's 128
                float bv[4] = {0.f, 0.f, 0.f, 0.f};
                if (bias) {
#pragma unroll
                    for (int r = 0; r < 4; r++)
                        if (wcol0 + cl + r < N) bv[r] = load_bias<C_DT>(bias, wcol0 + cl + r);
                }
#pragma unroll
                for (int ti = 0; ti < 4; ti++) {
                    const float v0 = acc[tj][ti][4 * g + 0] * inv + bv[0];
                    const float v1 = acc[tj][ti][4 * g + 1] * inv + bv[1];
                    const float v2 = acc[tj][ti][4 * g + 2] * inv + bv[2];
                    const float v3 = acc[tj][ti][4 * g + 3] * inv + bv[3];
                    *(uint2*)(ep + (ti * 32 + lm) * EPI_PITCH + cl * 2) = make_uint2(pack2<C_DT>(v0, v1), pack2<C_DT>(v2, v3));
                }
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own wave's tile only: no workgroup barrier needed
        uint16_t* Ch = (uint16_t*)C;
        const int chunk = lane & 15, rsub = lane >> 4;
        const int col = wcol0 + chunk * 8;
#pragma unroll 4
        for (int it = 0; it < 32; it++) {
            const int rl = it * 4 + rsub;
            const int row = wrow0 + rl;
            const uint4 v = *(const uint4*)(ep + rl * EPI_PITCH + chunk * 16);
            if (row < M && col < N) {
                uint16_t* dst = Ch + (int64_t)row * ldc + col;
                if (c_vec_ok && col + 8 <= N) {
                    store16_any(dst, v);
                } else {
                    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (col + i < N) dst[i] = (uint16_t)((w[i >> 1] >> (16 * (i & 1))) & 0xffffu);
                }
            }
        }
    }
}

// Raises a kernel's dynamic LDS limit once per device (the attribute is per device, calls may come from any
// host thread: a repeated call is harmless, a missing one is not).
template <typename K>
static int allow_big_lds(K kern, int bytes, std::atomic<uint64_t>& done_mask) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return check_hip(e, "hipGetDevice");
    const uint64_t bit = 1ull << (dev & 63);
    if (done_mask.load(std::memory_order_acquire) & bit) return 0;
    e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return check_hip(e, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
    done_mask.fetch_or(bit, std::memory_order_release);
    return 0;
}

// Both for 2-byte outputs with rows at odd multiples of two bytes (f8mi_gemm_dma16_odd.hip, f8mi_gemm_mid_odd.hip).
int launch_gemm_mid_odd(int a_fmt, int b_fmt, int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                        const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                        int64_t ldc, const void* bias, int c_vec_ok);
int launch_gemm_dma16_odd(int a_fmt, int b_fmt, int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                          const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb,
                          void* C, int64_t ldc, const void* bias, int tiles_m, int tiles_n, int c_vec_ok);
// Both, large and 128-row tiles, with the bias added to the rounded product (f8mi_gemm_biased.hip): operands as they are, e4m3.
// large: tiles of 256 x `cols` (256, 224); else 128 x cols (128, 256).
int launch_gemm_biased(bool large, int cols, int c_dtype, hipStream_t stream, const uint8_t* A, int64_t a_unit, const uint8_t* Bt, int64_t b_unit, int M, int N,
                       int K, const float* sa, const float* sb, void* C, int64_t ldc, const void* bias, int bias_fp32, int c_vec_ok);
// Tiles of 256 x 224 (f8mi_gemm_dma16_narrow.hip), rows of C at multiples of four bytes or fp32.
int launch_gemm_dma16_narrow(int a_fmt, int b_fmt, int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                             const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb,
                             void* C, int64_t ldc, const void* bias, int tiles_m, int tiles_n, int c_vec_ok);
// The 16x16x128 kernel with Bt (nt) or both operands (tt) given transposed: memory holds [contraction][rows];
// lda / ldb = bytes between contraction rows, a_unit / b_unit = bytes between blocks of 64 rows.
// 128-row-tile kernels (f8mi_gemm_mid_impl.h) for outputs of few 256 x 256 tiles: K % 128 == 0, aligned operands.
// wide = false: 128 x 128 tiles, true: 128 x 256.
int launch_gemm_mid(int a_fmt, int b_fmt, int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                    const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                    int64_t ldc, const void* bias, int c_vec_ok);
// They take over while their own tiles number at most one per CU (with more, the large tiles win again: measured):
// 128 x 128 tiles while at most 256 of them cover the output, else 128 x 256 tiles while 256 of those do.
// Returns 0: large tiles, 1: 128 x 128, 2: 128 x 256.
inline int use_mid_tiles(int64_t m, int64_t n, int64_t k) {
    if (k % 128 != 0 || k < 128) return 0;
    const int64_t row_tiles = (m + 127) / 128;
    if (row_tiles * ((n + 127) / 128) <= 256) return 1;
    if (row_tiles * ((n + 255) / 256) <= 256) return 2;
    return 0;
}
// few-row kernel (f8mi_gemm_skinny.hip): m <= SKINNY_MAX_M, K % 128 == 0, aligned operands.
constexpr int SKINNY_MAX_M = 256;
// Time estimates in us behind the choice between the few-row kernel, a round of 128-row tiles, and the same tiles
// with k split over workgroups.  They were fitted to earlier forms of these kernels and rank them, no more.  As the kernels are now,
// weights cold (rows, n x k: few-row / tiles / k split 8, 4 or 2 ways): 128, 8192 x 8192: 30 / 38 / 24; 128, 28672 x 8192: 110 / 46;
// 64, 28672 x 8192: 72 / 39; 64, 4096 x 14336: 30 / 45 / 20; 192, 4096 x 4096: 15.4 / 17.6 / 17.8; 4096 x 14336: 40 / 49 / 24; 8192 x
// 8192: 50 / 32 / 26; 14336 x 4096: 54 / 20; 28672 x 8192: 162 / 56.  Of 820 sizes with 17 - 1024 rows, n and k from 512 to 57344 and 28672,
// the choice is within 5 % of the best of the three in 671.  Where it is not, the few-row kernel is kept for narrow weights with a
// long k that a split would take in half the time (128, 512 x 28672: 67 / 71 / 20; 64, 2048 x 14336: 29 / 49 / 16), and tiles for 17 - 64 rows
// with k = 512 that the few-row kernel takes in two thirds of it (17, 4096 x 512: 3.5 / 6.0).
// They depend on the shape only, so the row-major and the k-blocked entry point decide alike.
//
// Few-row kernel: Bt at 6.5 TB/s from memory plus A (n / 32 workgroups x 16 row_tiles x k bytes) at 20 TB/s from L2,
// once per 128 rows; slower when its n / 32 workgroups per pass leave CUs idle.
inline double skinny_time_us(int64_t m, int64_t n, int64_t k) {
    const double passes = (double)((m + 127) / 128);
    const double row_tiles = m > 128 ? 8.0 : (double)((m + 15) / 16);  // 16-row tiles of A per pass
    const double wgs = passes * (double)((n + 31) / 32);
    const double idle = wgs < 256.0 ? __builtin_sqrt(256.0 / wgs) : 1.0;
    return passes * (2.0 + (double)n * (double)k * (0.154 + 0.025 * row_tiles) * 1e-6 * idle);
}
// Tiles: a round of 128 x 128 tiles was taken to cost 4.4 ns per unit of k, of 128 x 256 tiles 7.8 ns, of 256 x 256 tiles 10.6 ns, for
// 1 row or 128 (128 x 128 now: 5 us and 2.3 ns with few tiles, 4.2 with 128 and more; 128 x 256: 6 us and 6 - 7.3 ns).
inline double tiles_time_us(int64_t m, int64_t n, int64_t k) {
    const int64_t rt = (m + 127) / 128;
    if (rt * ((n + 127) / 128) <= 256) return 4.4e-3 * (double)k;
    if (rt * ((n + 255) / 256) <= 256) return 7.8e-3 * (double)k;
    return 10.6e-3 * (double)k * (double)((((m + 255) / 256) * ((n + 255) / 256) + 255) / 256);
}
// Up to 16 rows the few-row kernel always runs: it streams Bt once at memory speed.
inline bool use_skinny(int64_t m, int64_t n, int64_t k) {
    if (m > SKINNY_MAX_M || k <= 0 || k % 128 != 0) return false;
    if (m <= 16) return true;
    // With 33 - 128 rows the few-row kernel has one workgroup on a CU: more than 256 of them run in turn, and tiles are faster (us, few-row /
    // tiles: 33 rows, 8320 x 1024: 8.4 / 7.8, 9216 x 4096: 17.6 / 16.3; 48 rows, 10240 x 3072: 17.9 / 14.4; 64 rows, 14336 x 4096: 22.1 / 19.0; 96
    // rows, 14336 x 2048: 20.5 / 12.9; with 256: 48 rows, 8192 x 3072: 10.4 / 13.9, 8192 x 8192: 20.4 / 29.6).
    if (m > 32 && m <= 128 && n > 8192 && use_mid_tiles(m, n, k)) return false;
    return skinny_time_us(m, n, k) <= tiles_time_us(m, n, k);
}
// An output of at most 128 of the 128-row tiles and a long k: with `ws_bytes` of scratch for the partial sums, k is
// split 2, 4 or 8 ways so that (nearly) every CU gets a part, and a second kernel adds the parts in a fixed order.
// Returns the number of parts, 0 for no split.  Cost of the split: the parts written and read once (5 TB/s) and a launch.
inline int pick_k_splits(int64_t m, int64_t n, int64_t k, int64_t ws_bytes) {
    const int mode = use_mid_tiles(m, n, k);
    if (!mode || n % 4 != 0 || m <= 16 || ws_bytes <= 0) return 0;
    const int64_t tiles = ((m + 127) / 128) * ((n + (mode == 1 ? 127 : 255)) / (mode == 1 ? 128 : 256));
    if (tiles > 128) return 0;
    const double t_round = (mode == 1 ? 4.4e-3 : 7.8e-3) * (double)k;
    const double t_skinny = m <= SKINNY_MAX_M ? skinny_time_us(m, n, k) : 1e30;
    const double t_other = t_skinny < t_round ? t_skinny : t_round;
    int best = 0;
    double t_best = 0.9 * t_other;  // the estimates are not better than that
    for (int s = 2; s <= 8; s *= 2) {
        if (tiles * s > 256 || k % (128 * s) != 0 || k / s < 1024 || (int64_t)s * m * n * 4 > ws_bytes) break;
        const double t = t_round / s + 3.0 + (double)s * (double)m * (double)n * 8.0 / 5e6 + 4.0;
        if (t < t_best) { t_best = t; best = s; }
    }
    return best;
}
int launch_gemm_mid_splitk(int a_fmt, int b_fmt, int c_dtype, bool wide, int k_splits, float* partial, hipStream_t stream, const uint8_t* A,
                           int64_t lda, int64_t a_unit, const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa,
                           const float* sb, void* C, int64_t ldc, const void* bias, int c_vec_ok);
int launch_gemm_skinny(int a_fmt, int b_fmt, int c_dtype, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                       const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                       int64_t ldc, const void* bias);
// The 128-row-tile kernel on the same transposed operands (f8mi_gemm_mid_nt.hip, f8mi_gemm_mid_tt.hip).
int launch_gemm_mid_nt(int a_fmt, int b_fmt, int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                       const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                       int64_t ldc, const void* bias, int c_vec_ok);
int launch_gemm_mid_tt(int a_fmt, int b_fmt, int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                       const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                       int64_t ldc, const void* bias, int c_vec_ok);
int launch_gemm_dma16_nt(int a_fmt, int b_fmt, int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                         const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb,
                         void* C, int64_t ldc, const void* bias, int tiles_m, int tiles_n, int c_vec_ok);
int launch_gemm_dma16_tt(int a_fmt, int b_fmt, int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                         const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb,
                         void* C, int64_t ldc, const void* bias, int tiles_m, int tiles_n, int c_vec_ok);

// LDS-DMA kernel (f8mi_gemm_dma.hip).  Needs 16-byte aligned operands and strides and K % 64 == 0, K >= 384.
// lda / ldb: bytes between operand rows, a_unit / b_unit: bytes between 64-deep units of one row
// (row-major: (row stride, 64); k-blocked [K/64][rows][64]: (64, rows * 64)).
int launch_gemm_dma(int a_fmt, int b_fmt, int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                    const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb,
                    void* C, int64_t ldc, const void* bias, int tiles_m, int tiles_n, int c_vec_ok);
// The same on the 16x16x128 MFMA (f8mi_gemm_dma16.hip); additionally needs K % 128 == 0.
int launch_gemm_dma16(int a_fmt, int b_fmt, int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                      const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb,
                      void* C, int64_t ldc, const void* bias, int tiles_m, int tiles_n, int c_vec_ok);

}  // namespace f8mi
