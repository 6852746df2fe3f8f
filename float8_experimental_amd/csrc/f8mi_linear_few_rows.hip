// A linear of at most 16 rows and F8MI_FEW_ROWS_ELEMS activations in one kernel: every workgroup casts the activations to
// e4m3 itself, into its LDS, while the first weights are on their way.  HBM-bound: the weight, one byte per element, is all
// that has to be read.
//
// As two launches (cast, few-row GEMM) the one in front costs a third of a decode step of one linear: 1 x 8192 -> 8192: 20.3 ->
// 15.5 us (weights cold; reading them at 7 TB/s: 9.6), 1 x 4096 -> 4096: 9.7 -> 7.0, 8 x 4096 -> 4096: 12.3 -> 9.6, 4 x 8192 ->
// 28672: 52.5 -> 50.3.
//
// A workgroup of eight waves holds x in registers (at most 64 elements a lane), finds its maximum (dynamic scaling; the
// scale is given otherwise), casts and parks the bytes in LDS.  It owns 16 NT columns of C; the waves split k eight ways and
// stream their part of the weight into MFMA operands (two 16-byte loads per lane and 128-deep step), DEPTH steps in flight,
// a slot refilled as soon as it has been multiplied; the eight partial sums meet in LDS and are added in a fixed order.
// Split, order of steps and order of the sums are those of f8mi_gemm_skinny.hip, the arithmetic of the cast that of
// f8mi_cast.hip: the same bits.
//
// More activations than that are cast by a launch of their own: the conversion is a few vector instructions per element and
// lane, and every workgroup would repeat it (16 x 8192 -> 8192: 25 us that way for a product of 16).
#include "f8mi_cast_util.h"
#include "f8mi_gemm_util.h"

namespace f8mi {

typedef float v4f_l __attribute__((ext_vector_type(4)));

constexpr int FR_WAVES = 8;
constexpr int FR_THREADS = FR_WAVES * 64;
constexpr int FR_MAX_M = 16;
// Steps in flight per wave: at most what the registers next to x allow (128 a lane, with two workgroups a CU; fp32 x takes 64 of them)
constexpr int fr_depth(int nt, int dt) { return nt == 2 && dt == F8MI_FP32 ? 2 : 4; }
constexpr int FR_LDS_PAD = 16;  // bytes between rows of x8 in LDS

__device__ __forceinline__ v8i fr_load_weight(const uint8_t* p) {
    const uint4 lo = *(const uint4*)p, hi = *(const uint4*)(p + 16);
    return (v8i){(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
}

// 16 bytes of x: EPV elements -> EPV e4m3 bytes (the upper word unused for fp32)
template <int DT, int PROD>
__device__ __forceinline__ uint2 cast_piece(uint4 q, float scale) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    uint32_t r[2] = {0u, 0u};
#pragma unroll
    for (int i = 0; i < (DT == F8MI_FP32 ? 1 : 2); i++) {
        float e[4], f[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if constexpr (DT == F8MI_FP32) e[j] = __uint_as_float(w[j]);
            else {
                const uint32_t h = (j & 1) ? w[2 * i + j / 2] >> 16 : w[2 * i + j / 2] & 0xffffu;
                e[j] = DT == F8MI_BF16 ? bf16_bits_to_float(h) : fp16_bits_to_float(h);
            }
        }
        scale_clamp2<PROD>(e[0], e[1], scale, 448.0f, f[0], f[1]);
        scale_clamp2<PROD>(e[2], e[3], scale, 448.0f, f[2], f[3]);
        r[i] = cvt4_fp8<F8MI_E4M3FN>(f[0], f[1], f[2], f[3]);
    }
    return make_uint2(r[0], r[1]);
}

template <int DT>
__device__ __forceinline__ uint32_t absmax16bytes(uint4 v, uint32_t m) {  // 16-bit types: two maxima side by side
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if constexpr (DT == F8MI_FP32) m = max(m, w[i] & 0x7fffffffu);
        else m = absmax16x2(w[i], m);
    }
    return m;
}

template <int DT, int PROD, int BF, int NT, int DEPTH>
__global__ __launch_bounds__(FR_THREADS, 4) void linear_few_rows_kernel(
    const uint8_t* __restrict__ x, int64_t ldx, const uint8_t* __restrict__ Bt, int64_t ldb, int64_t b_unit, int M, int N, int K,
    const float* __restrict__ sx_dev, const float* __restrict__ sb_dev, void* __restrict__ C, int64_t ldc, const void* __restrict__ bias) {
    constexpr int ESZ = DT == F8MI_FP32 ? 4 : 2, EPV = 16 / ESZ;
    constexpr int PIECES = F8MI_FEW_ROWS_ELEMS / EPV / FR_THREADS;
    extern __shared__ __align__(16) uint8_t x8[];  // [M][K + FR_LDS_PAD]
    __shared__ float4 part[FR_WAVES / 2][NT][64];
    __shared__ uint32_t red[FR_WAVES];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lm = lane & 15, lq = lane >> 4;
    const int n0 = blockIdx.x * (16 * NT);
    const int steps = K / 128, pitch = K + FR_LDS_PAD;
    const int s0 = steps * wave / FR_WAVES, s1 = steps * (wave + 1) / FR_WAVES;
    const float sb = *sb_dev;

    // x, ahead of the weights: needed first.  K % 128 == 0: rows are whole 16-byte pieces
    const uint32_t per_row = (uint32_t)K / EPV, items = (uint32_t)M * per_row;
    uint4 v[PIECES];
#pragma unroll
    for (int u = 0; u < PIECES; u++) {
        const uint32_t i = u * FR_THREADS + threadIdx.x;
        v[u] = make_uint4(0u, 0u, 0u, 0u);
        if (i < items) {
            const uint32_t row = i / per_row;
            const u32x4 t = *(const u32x4_any*)(x + (row * ldx + (int64_t)(i - row * per_row) * EPV) * ESZ);
            v[u] = make_uint4(t.x, t.y, t.z, t.w);
        }
    }
    // a lane's 32 bytes of step s: row * ld + (2s + lq / 2) * unit + 32 * (lq % 2); rows past the end re-read the last one.  Next to fp32 x
    // the wave's part of the address is scalar and the lane's 32 bits (the host has checked that they do): with a 64-bit pointer per
    // lane 32 columns spilled, and one step in flight instead of two cost more on long k (1 row, 14336 x 32768: 88.9 us with one, 83.2
    // with two).  16-bit x leaves the registers for pointers, which are faster (1 row, 8192 x 8192, weights in cache: 13.2 / 12.7 us).
    constexpr bool SCALAR_BASE = DT == F8MI_FP32;
    const uint8_t* const base = Bt + (int64_t)n0 * ldb;
    const uint8_t* pb[NT];
    uint32_t off[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
        if constexpr (SCALAR_BASE) off[nt] = (uint32_t)(min(nt * 16 + lm, N - 1 - n0) * ldb + (lq >> 1) * b_unit + (lq & 1) * 32);
        else pb[nt] = Bt + (int64_t)min(n0 + nt * 16 + lm, N - 1) * ldb + (lq >> 1) * b_unit + (lq & 1) * 32;
    }
    v8i fb[DEPTH][NT];
    auto load = [&](int d, int s) __attribute__((always_inline)) {  // past the wave's range: a valid address, the product is skipped
        const int sd = min(s, s1 - 1);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            if constexpr (SCALAR_BASE) fb[d][nt] = fr_load_weight(base + 2 * (int64_t)sd * b_unit + off[nt]);
            else fb[d][nt] = fr_load_weight(pb[nt] + 2 * (int64_t)sd * b_unit);
        }
    };
    if (s0 < s1) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) load(d, s0 + d);
    }

    float scale;
    if (sx_dev) {
        scale = *sx_dev;
    } else {
        uint32_t m = 0;
#pragma unroll
        for (int u = 0; u < PIECES; u++) m = absmax16bytes<DT>(v[u], m);
        if constexpr (DT != F8MI_FP32) m = fold16(m);
        m = wave_max_u32(m);
        if (lane == 0) red[wave] = m;
        lds_barrier();  // (does not wait for the weights)
        m = red[0];
#pragma unroll
        for (int i = 1; i < FR_WAVES; i++) m = max(m, red[i]);
        scale = amax_to_scale_dev(abs_bits_to_float(m, DT), DT, F8MI_E4M3FN, DT == F8MI_FP16);
    }
#pragma unroll
    for (int u = 0; u < PIECES; u++) {
        const uint32_t i = u * FR_THREADS + threadIdx.x;
        if (i < items) {
            const uint32_t row = i / per_row;
            const uint2 c = cast_piece<DT, PROD>(v[u], scale);
            uint8_t* dst = x8 + row * pitch + (i - row * per_row) * EPV;
            if constexpr (DT == F8MI_FP32) *(uint32_t*)dst = c.x;
            else *(uint2*)dst = c;
        }
    }
    lds_barrier();
    const uint8_t* px = x8 + min(lm, M - 1) * pitch + lq * 32;

    v4f_l acc[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) acc[nt] = (v4f_l){0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int d, int s) __attribute__((always_inline)) {
        const v8i fa = read_frag(px + s * 128, px + s * 128 + 16);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[nt] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[d][nt], fa, acc[nt], BF, F8MI_E4M3FN, 0, 0, 0, 0);
    };
    int s = s0;
    for (; s + DEPTH < s1; s += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            multiply(d, s + d);
            load(d, s + DEPTH + d);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; d++)
        if (s + d < s1) multiply(d, s + d);

    // the eight partial sums of every output: waves 4..7 hand theirs to waves 0..3, then the four sums are added in a fixed order
    if (wave >= FR_WAVES / 2) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) part[wave - FR_WAVES / 2][nt][lane] = make_float4(acc[nt][0], acc[nt][1], acc[nt][2], acc[nt][3]);
    }
    __syncthreads();
    if (wave < FR_WAVES / 2) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const float4 p = part[wave][nt][lane];
            part[wave][nt][lane] = make_float4(acc[nt][0] + p.x, acc[nt][1] + p.y, acc[nt][2] + p.z, acc[nt][3] + p.w);
        }
    }
    __syncthreads();
    if (threadIdx.x >= NT * 64) return;
    const int tile = wave;
    float4 sum = part[0][tile][lane];
#pragma unroll
    for (int w = 1; w < FR_WAVES / 2; w++) {
        const float4 p = part[w][tile][lane];
        sum.x += p.x; sum.y += p.y; sum.z += p.z; sum.w += p.w;
    }
    // MFMA(first = weight rows, second = rows of x): lane l holds row l % 16 of x and columns 4 * (l / 16) + e
    const float inv = __fdiv_rn(1.0f, scale) * __fdiv_rn(1.0f, sb);
    const int col = n0 + tile * 16 + 4 * lq;
    if (lm >= M) return;
    const float t[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        if (col + e >= N) break;
        const float r = t[e] * inv + (bias ? load_bias<DT>(bias, col + e) : 0.f);
        const int64_t at = (int64_t)lm * ldc + col + e;
        if constexpr (DT == F8MI_FP32) ((float*)C)[at] = r;
        else ((uint16_t*)C)[at] = (uint16_t)(pack2<DT>(r, 0.f) & 0xffffu);
    }
}

struct FewRowsArgs {
    const uint8_t* x; int64_t ldx; const uint8_t* w; int64_t ldb, b_unit; int M, N, K;
    const float* sx; const float* sb; void* C; int64_t ldc; const void* bias;
};
template <int DT, int PROD, int BF, int NT, int DEPTH>
static int launch_fr4(hipStream_t stream, const FewRowsArgs& a) {
    hipLaunchKernelGGL((linear_few_rows_kernel<DT, PROD, BF, NT, DEPTH>), dim3((unsigned)((a.N + 16 * NT - 1) / (16 * NT))), dim3(FR_THREADS), (size_t)a.M * (a.K + FR_LDS_PAD), stream,
                       a.x, a.ldx, a.w, a.ldb, a.b_unit, a.M, a.N, a.K, a.sx, a.sb, a.C, a.ldc, a.bias);
    return check_hip(hipGetLastError(), "few-row linear kernel launch");
}
template <int DT, int PROD, int BF, int NT>
static int launch_fr3(hipStream_t stream, const FewRowsArgs& a) {
    // no more slots than a wave has steps, as in f8mi_gemm_skinny.hip (1 row, 131072 x 512: 36.9 / 24.0 us; 8 rows, 8192 x 1024: 7.1 / 6.5)
    constexpr int DEPTH = fr_depth(NT, DT);
    const int steps = (a.K / 128 + FR_WAVES - 1) / FR_WAVES;
    if constexpr (DEPTH > 1)
        if (steps <= 1) return launch_fr4<DT, PROD, BF, NT, 1>(stream, a);
    if constexpr (DEPTH > 2)
        if (steps <= 2) return launch_fr4<DT, PROD, BF, NT, 2>(stream, a);
    return launch_fr4<DT, PROD, BF, NT, DEPTH>(stream, a);
}
template <int DT, int PROD, int BF>
static int launch_fr2(hipStream_t stream, const FewRowsArgs& a) {
    // 32 columns a workgroup where that leaves every CU with one (each converts all of x), else 16: 1 row, 8192 x 8192: 17.3 / 15.5
    // us with 32 / 16; 14336 x 4096: 13.5 / 16.5; 4 rows, 28672 x 8192: 50.3 with 32
    if (a.N > 32 * cu_count()) return launch_fr3<DT, PROD, BF, 2>(stream, a);
    return launch_fr3<DT, PROD, BF, 1>(stream, a);
}
template <int DT, int PROD>
static int launch_fr1(int w_fmt, hipStream_t stream, const FewRowsArgs& a) {
    return w_fmt == F8MI_E4M3FN ? launch_fr2<DT, PROD, F8MI_E4M3FN>(stream, a) : launch_fr2<DT, PROD, F8MI_E5M2>(stream, a);
}

}  // namespace f8mi

using namespace f8mi;

extern "C" int f8mi_linear_few_rows(const void* x, int64_t ldx, int dtype, const float* scale_x_dev, int product_dtype, const void* w, int w_fmt,
                                    int w_layout, const float* scale_w_dev, int64_t m, int64_t n, int64_t k, void* c, int64_t ldc,
                                    const void* bias_dev, void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (dtype < 0 || dtype > 2 || w_fmt < 0 || w_fmt > 1) { set_error("f8mi_linear_few_rows: unknown dtype/format code"); return F8MI_ERR_INVALID_ARG; }
    if (scale_x_dev && product_dtype != dtype && product_dtype != F8MI_FP32) { set_error("f8mi_linear_few_rows: product_dtype must be the input dtype or fp32"); return F8MI_ERR_INVALID_ARG; }
    if (m < 0 || n < 0 || k < 0 || ldx < k || ldc < n) { set_error("f8mi_linear_few_rows: bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k); return F8MI_ERR_INVALID_ARG; }
    if (m == 0 || n == 0) return F8MI_OK;
    if (m > FR_MAX_M || k < 128 || k % 128 != 0 || m * k > F8MI_FEW_ROWS_ELEMS || n > (w_layout && dtype == F8MI_FP32 ? 0x3ffff00LL : 0x7fffff00LL) || (w_layout != F8MI_LAYOUT_ROWMAJOR && w_layout != F8MI_LAYOUT_KBLOCK64) || (uintptr_t)w % 16 != 0) { set_error("f8mi_linear_few_rows: at most 16 rows and 32768 activations, k a multiple of 128, a 16-byte aligned row-major or k-blocked weight (m=%lld k=%lld layout=%d)", (long long)m, (long long)k, w_layout); return F8MI_ERR_UNSUPPORTED; }
    if (!x || !w || !scale_w_dev || !c) { set_error("f8mi_linear_few_rows: null pointer"); return F8MI_ERR_INVALID_ARG; }
    FewRowsArgs a{(const uint8_t*)x, ldx, (const uint8_t*)w, w_layout ? 64 : k, w_layout ? n * 64 : 64, (int)m, (int)n, (int)k, scale_x_dev,
                  scale_w_dev, c, ldc, bias_dev};
    ProfScope prof(F8MI_K_GEMM, 2.0 * (double)m * (double)n * (double)k, stream);
    const bool wide_product = scale_x_dev && product_dtype == F8MI_FP32;
    if (dtype == F8MI_BF16) return wide_product ? launch_fr1<F8MI_BF16, F8MI_FP32>(w_fmt, stream, a) : launch_fr1<F8MI_BF16, F8MI_BF16>(w_fmt, stream, a);
    if (dtype == F8MI_FP16) return wide_product ? launch_fr1<F8MI_FP16, F8MI_FP32>(w_fmt, stream, a) : launch_fr1<F8MI_FP16, F8MI_FP16>(w_fmt, stream, a);
    return launch_fr1<F8MI_FP32, F8MI_FP32>(w_fmt, stream, a);
}
