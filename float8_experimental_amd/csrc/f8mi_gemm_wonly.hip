// Weight-only inference: C[m][n] = sum_k x[m][k] * round(w8[n][k] / scale), x and the dequantised weight in bf16 / fp16 /
// fp32, fp32 accumulation.  HBM-bound for few rows: the fp8 weight, one byte per element, is all that has to be read.
//
// Dequantising into a tensor first reads n k, writes 2 n k, reads 2 n k and divides element by element: 14336 x 4096 took
// 143 us (conversion) + 149 us (division) + 20 us (library GEMM) for four tokens, now 16.5 us in all (reading the weight at
// 7 TB/s: 8.4; what is left is launch and ramp, and the conversions, which the few waves per SIMD do not all hide).  Here the weight goes from memory to
// registers, is dequantised there and multiplied, as in the few-row fp8 kernel: a workgroup of eight waves owns 16 NT columns
// of C and 16 MT rows, the waves split k eight ways, a lane's load is 16 consecutive k bytes of one weight row and the
// same 16 elements of one row of x (from the L2), which are two operands of v_mfma_f32_16x16x32_bf16 (f16) or sixteen of
// v_mfma_f32_16x16x4_f32 -- the instruction's own order of k inside a step does not matter as long as both operands use the
// same.  The eight partial sums meet in LDS and are added in a fixed order.
//
// The quotient has to be the one torch's division gives, fp32 and then rounded to the tensor's type.  A division is ten
// instructions, twice what the memory rate leaves time for; an fp8 format has only 128 magnitudes, so every wave first
// checks, two codes per lane, that a product with the reciprocal (fp32: with one Newton step on the remainder) gives the
// same bits for ALL of them, and divides only where one differs.
//
// Rows of w and x start at any multiple of the element size (16-byte loads at any alignment, see f8mi_common.h); a k that
// is no multiple of 64 ends in one guarded step, which the last wave takes.
#include "f8mi_gemm_util.h"

namespace f8mi {

typedef float v4f_w __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf_w __attribute__((ext_vector_type(8)));
typedef _Float16 v8h_w __attribute__((ext_vector_type(8)));

constexpr int WO_WAVES = 8;
constexpr int WO_THREADS = WO_WAVES * 64;
constexpr int WO_STEP = 64;  // k elements per step: 4 lanes x 16

// sixteen consecutive elements of a row of x / of the dequantised weight, as they sit in the dtype
template <int DT>
struct Elems16 {
    uint32_t w[DT == F8MI_FP32 ? 16 : 8];
};

template <int DT>
__device__ __forceinline__ void load16(Elems16<DT>& r, const uint8_t* p) {
#pragma unroll
    for (int i = 0; i < (DT == F8MI_FP32 ? 4 : 2); i++) {
        const u32x4 v = *(const u32x4_any*)(p + 16 * i);
        r.w[4 * i] = v.x; r.w[4 * i + 1] = v.y; r.w[4 * i + 2] = v.z; r.w[4 * i + 3] = v.w;
    }
}

// the first `valid` of the sixteen, zeros behind them
template <int DT>
__device__ __forceinline__ void load16_tail(Elems16<DT>& r, const uint8_t* p, int valid) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
        if constexpr (DT == F8MI_FP32) {
            r.w[i] = i < valid ? ((const uint32_t*)p)[i] : 0u;
        } else {
            const uint32_t h = i < valid ? ((const uint16_t*)p)[i] : 0u;
            if (i & 1) r.w[i >> 1] |= h << 16;
            else r.w[i >> 1] = h;
        }
    }
}

template <int FMT>
__device__ __forceinline__ void widen2(uint32_t w, bool hi, float& a, float& b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    f2 r;
    if constexpr (FMT == F8MI_E4M3FN) r = hi ? __builtin_amdgcn_cvt_pk_f32_fp8(w, true) : __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
    else r = hi ? __builtin_amdgcn_cvt_pk_f32_bf8(w, true) : __builtin_amdgcn_cvt_pk_f32_bf8(w, false);
    a = r.x;
    b = r.y;
}

// v / s in fp32.  FAST: by the reciprocal (only used where it gives the same bits for every code of the format)
template <int DT, bool FAST>
__device__ __forceinline__ float quotient(float v, float s, float rcp) {
    if constexpr (!FAST) return __fdiv_rn(v, s);
    else if constexpr (DT != F8MI_FP32) {
        float q = __fmul_rn(v, rcp);
        asm("" : "+v"(q));  // rounded to fp32 here: not folded with the conversion behind it into one rounding
        return q;
    } else {
        const float q = __fmul_rn(v, rcp);
        return __fmaf_rn(__fmaf_rn(-q, s, v), rcp, q);
    }
}

// the bits of the quotient in the dtype
template <int DT, bool FAST>
__device__ __forceinline__ uint32_t quotient_bits(float v, float s, float rcp) {
    const float q = quotient<DT, FAST>(v, s, rcp);
    if constexpr (DT == F8MI_FP32) return __float_as_uint(q);
    else return pack2<DT>(q, 0.f) & 0xffffu;
}

template <int FMT, int DT>
__device__ __forceinline__ bool fast_ok(float s, float rcp) {
    bool same = true;
#pragma unroll
    for (int h = 0; h < 2; h++) {
        float v, unused;
        widen2<FMT>((threadIdx.x & 63) + 64u * h, false, v, unused);
        const uint32_t a = quotient_bits<DT, true>(v, s, rcp), b = quotient_bits<DT, false>(v, s, rcp);
        same = same && (a == b || v != v);  // (in fp32 the remainder of an infinity is NaN: e5m2 divides there)
    }
    return __all(same);
}

template <int FMT, int DT, bool FAST>
__device__ __forceinline__ void dequant16(Elems16<DT>& r, uint4 w, float s, float rcp) {
    const uint32_t in[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        float f[4];
        widen2<FMT>(in[i], false, f[0], f[1]);
        widen2<FMT>(in[i], true, f[2], f[3]);
#pragma unroll
        for (int j = 0; j < 4; j++) f[j] = quotient<DT, FAST>(f[j], s, rcp);
        if constexpr (DT == F8MI_FP32) {
#pragma unroll
            for (int j = 0; j < 4; j++) r.w[4 * i + j] = __float_as_uint(f[j]);
        } else {
            r.w[2 * i] = pack2<DT>(f[0], f[1]);
            r.w[2 * i + 1] = pack2<DT>(f[2], f[3]);
        }
    }
}

template <int DT>
__device__ __forceinline__ v4f_w mma16(const Elems16<DT>& b, const Elems16<DT>& a, v4f_w acc) {
    if constexpr (DT == F8MI_FP32) {
#pragma unroll
        for (int i = 0; i < 16; i++)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(b.w[i]), __uint_as_float(a.w[i]), acc, 0, 0, 0);
    } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const u32x4 bw = {b.w[4 * h], b.w[4 * h + 1], b.w[4 * h + 2], b.w[4 * h + 3]};
            const u32x4 aw = {a.w[4 * h], a.w[4 * h + 1], a.w[4 * h + 2], a.w[4 * h + 3]};
            if constexpr (DT == F8MI_BF16) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf_w, bw), __builtin_bit_cast(v8bf_w, aw), acc, 0, 0, 0);
            else acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h_w, bw), __builtin_bit_cast(v8h_w, aw), acc, 0, 0, 0);
        }
    }
    return acc;
}

// Steps in flight per wave.  More of them cost more registers than they hide latency: what is in flight per CU is the waves'
// (14336 x 4096, 1 row: 16.6 us with two steps, 19.2 with four, 23.8 with six; 4096 x 14336: 15.7 / 14.9 / 16.2).
constexpr int wo_depth(int mt) { return mt == 4 ? 1 : 2; }

template <int DT, int MT, int NT>
struct WonlyBatch {
    static constexpr int DEPTH = wo_depth(MT);
    uint4 w[DEPTH][NT];
    Elems16<DT> x[DEPTH][MT];
    // step st into slot d; past the wave's range a valid address (the product is skipped)
    __device__ __forceinline__ void load(const uint8_t* const (&px)[MT], const uint8_t* const (&pw)[NT], int d, int st, int s1) {
        const int64_t k = (int64_t)min(st, s1 - 1) * WO_STEP;
#pragma unroll
        for (int nt = 0; nt < NT; nt++) w[d][nt] = load_nt16_any(pw[nt] + k);
#pragma unroll
        for (int mt = 0; mt < MT; mt++) load16<DT>(x[d][mt], px[mt] + k * (DT == F8MI_FP32 ? 4 : 2));
    }
    template <int FMT, bool FAST>
    __device__ __forceinline__ void multiply(int d, float s, float rcp, v4f_w (&acc)[MT][NT]) {
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            Elems16<DT> wd;
            dequant16<FMT, DT, FAST>(wd, w[d][nt], s, rcp);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt][nt] = mma16<DT>(wd, x[d][mt], acc[mt][nt]);
        }
    }
};

// One wave's part [s0, s1) of the full 64-deep steps, the first DEPTH of them on their way, and, if `tail` > 0, the guarded
// step of `tail` elements at `steps`.
template <int FMT, int DT, int MT, int NT, bool FAST>
__device__ __forceinline__ void wonly_accumulate(WonlyBatch<DT, MT, NT>& in, const uint8_t* const (&px)[MT], const uint8_t* const (&pw)[NT],
                                                 int s0, int s1, int steps, int tail, float s, float rcp, v4f_w (&acc)[MT][NT]) {
    constexpr int ESZ = DT == F8MI_FP32 ? 4 : 2;
    int st = s0;
    for (; st + in.DEPTH < s1; st += in.DEPTH) {  // a slot is filled again as soon as it has been multiplied
#pragma unroll
        for (int d = 0; d < in.DEPTH; d++) {
            in.template multiply<FMT, FAST>(d, s, rcp, acc);
            in.load(px, pw, d, st + in.DEPTH + d, s1);
        }
    }
#pragma unroll
    for (int d = 0; d < in.DEPTH; d++)
        if (st + d < s1) in.template multiply<FMT, FAST>(d, s, rcp, acc);
    if (tail > 0) {
        const int valid = min(max(tail - (int)((threadIdx.x & 63) >> 4) * 16, 0), 16);
        const int64_t k = (int64_t)steps * WO_STEP;
        Elems16<DT> x[MT];
#pragma unroll
        for (int mt = 0; mt < MT; mt++) load16_tail<DT>(x[mt], px[mt] + k * ESZ, valid);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            uint32_t b[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int i = 0; i < 16; i++)
                if (i < valid) b[i >> 2] |= (uint32_t)pw[nt][k + i] << (8 * (i & 3));
            Elems16<DT> wd;
            dequant16<FMT, DT, FAST>(wd, make_uint4(b[0], b[1], b[2], b[3]), s, rcp);
#pragma unroll
            for (int mt = 0; mt < MT; mt++) acc[mt][nt] = mma16<DT>(wd, x[mt], acc[mt][nt]);
        }
    }
}

template <int FMT, int DT, int MT, int NT>
__global__ __launch_bounds__(WO_THREADS) void gemm_wonly_kernel(const uint8_t* __restrict__ x, int64_t ldx, const uint8_t* __restrict__ w,
                                                                int64_t ldw, int M_all, int N, int K, const float* __restrict__ scale_dev,
                                                                uint8_t* __restrict__ C, int64_t ldc) {
    constexpr int ESZ = DT == F8MI_FP32 ? 4 : 2;
    const int m_base = blockIdx.y * (16 * MT);
    const int M = min(M_all - m_base, 16 * MT);
    __shared__ float4 part[WO_WAVES / 2][MT * NT][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lm = lane & 15, lq = lane >> 4;
    const int n0 = blockIdx.x * (16 * NT);
    const int steps = K / WO_STEP;
    const int s0 = (int)((int64_t)steps * wave / WO_WAVES), s1 = (int)((int64_t)steps * (wave + 1) / WO_WAVES);

    const uint8_t* px[MT];  // rows past the end re-read the last one
    const uint8_t* pw[NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++) px[mt] = x + ((int64_t)(m_base + min(mt * 16 + lm, M - 1)) * ldx + lq * 16) * ESZ;
#pragma unroll
    for (int nt = 0; nt < NT; nt++) pw[nt] = w + (int64_t)min(n0 + nt * 16 + lm, N - 1) * ldw + lq * 16;

    const float scale = *scale_dev;
    WonlyBatch<DT, MT, NT> in;  // on the way while the codes are checked
    if (s0 < s1) {
#pragma unroll
        for (int d = 0; d < in.DEPTH; d++) in.load(px, pw, d, s0 + d, s1);
    }
    v4f_w acc[MT][NT];
#pragma unroll
    for (int mt = 0; mt < MT; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = (v4f_w){0.f, 0.f, 0.f, 0.f};
    // the scale in the dtype the division takes place in: a 0-dim fp32 scale is rounded to the tensor's type first
    const float s = round_to<DT>(scale), rcp = __fdiv_rn(1.0f, s);
    const int tail = wave == WO_WAVES - 1 ? K - steps * WO_STEP : 0;
    if (fast_ok<FMT, DT>(s, rcp)) wonly_accumulate<FMT, DT, MT, NT, true>(in, px, pw, s0, s1, steps, tail, s, rcp, acc);
    else wonly_accumulate<FMT, DT, MT, NT, false>(in, px, pw, s0, s1, steps, tail, s, rcp, acc);

    if (wave >= WO_WAVES / 2) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++)
                part[wave - WO_WAVES / 2][mt * NT + nt][lane] = make_float4(acc[mt][nt][0], acc[mt][nt][1], acc[mt][nt][2], acc[mt][nt][3]);
    }
    __syncthreads();
    if (wave < WO_WAVES / 2) {
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const float4 p = part[wave][mt * NT + nt][lane];
                part[wave][mt * NT + nt][lane] = make_float4(acc[mt][nt][0] + p.x, acc[mt][nt][1] + p.y, acc[mt][nt][2] + p.z, acc[mt][nt][3] + p.w);
            }
    }
    __syncthreads();
    for (int item = threadIdx.x; item < MT * NT * 64; item += WO_THREADS) {
        const int tile = item >> 6, l = item & 63;
        float4 sum = part[0][tile][l];
#pragma unroll
        for (int v = 1; v < WO_WAVES / 2; v++) {
            const float4 p = part[v][tile][l];
            sum.x += p.x; sum.y += p.y; sum.z += p.z; sum.w += p.w;
        }
        // MFMA(first = weight rows, second = rows of x): lane l holds row l % 16 of x's tile and columns 4 * (l / 16) + e
        const int row = (tile / NT) * 16 + (l & 15);
        const int col = n0 + (tile % NT) * 16 + 4 * (l >> 4);
        if (row >= M) continue;
        const float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (col + e >= N) break;
            const int64_t at = (int64_t)(m_base + row) * ldc + col + e;
            if constexpr (DT == F8MI_FP32) ((float*)C)[at] = v[e];
            else ((uint16_t*)C)[at] = (uint16_t)(pack2<DT>(v[e], 0.f) & 0xffffu);
        }
    }
}

// The same dequantisation into a tensor, for more rows than one pass over the weight pays for: reads a byte and writes two
// (four) per element, in one launch.  HBM-bound.
template <int FMT, int DT, bool FAST>
__device__ __forceinline__ void dequant_chunk(const uint8_t* in, uint8_t* out, int64_t n, int64_t at, float s, float rcp) {
    constexpr int ESZ = DT == F8MI_FP32 ? 4 : 2;
    Elems16<DT> r;
    if (at + 16 <= n) {
        dequant16<FMT, DT, FAST>(r, load_nt16_any(in + at), s, rcp);
#pragma unroll
        for (int i = 0; i < (DT == F8MI_FP32 ? 4 : 2); i++)
            store16_any(out + at * ESZ + 16 * i, make_uint4(r.w[4 * i], r.w[4 * i + 1], r.w[4 * i + 2], r.w[4 * i + 3]));
        return;
    }
    for (int64_t e = at; e < n; e++) {
        float v, unused;
        widen2<FMT>(in[e], false, v, unused);
        const uint32_t b = quotient_bits<DT, FAST>(v, s, rcp);
        if constexpr (DT == F8MI_FP32) ((uint32_t*)out)[e] = b;
        else ((uint16_t*)out)[e] = (uint16_t)b;
    }
}

template <int FMT, int DT>
__global__ __launch_bounds__(256) void dequant_kernel(const uint8_t* __restrict__ in, int64_t n, const float* __restrict__ scale_dev,
                                                      uint8_t* __restrict__ out) {
    const float s = round_to<DT>(*scale_dev), rcp = __fdiv_rn(1.0f, s);
    const bool fast = fast_ok<FMT, DT>(s, rcp);
    const int64_t step = (int64_t)gridDim.x * 256 * 16;
    for (int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 16; at < n; at += step) {
        if (fast) dequant_chunk<FMT, DT, true>(in, out, n, at, s, rcp);
        else dequant_chunk<FMT, DT, false>(in, out, n, at, s, rcp);
    }
}

template <int FMT, int DT, int NT>
static int launch_wonly2(hipStream_t stream, const uint8_t* x, int64_t ldx, const uint8_t* w, int64_t ldw, int M, int N, int K,
                         const float* scale, uint8_t* C, int64_t ldc) {
    const unsigned gx = (unsigned)((N + 16 * NT - 1) / (16 * NT));
    const dim3 b(WO_THREADS);
    if (M <= 16) hipLaunchKernelGGL((gemm_wonly_kernel<FMT, DT, 1, NT>), dim3(gx), b, 0, stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
    else if (M <= 32) hipLaunchKernelGGL((gemm_wonly_kernel<FMT, DT, 2, NT>), dim3(gx), b, 0, stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
    else hipLaunchKernelGGL((gemm_wonly_kernel<FMT, DT, 4, NT>), dim3(gx, (unsigned)((M + 63) / 64)), b, 0, stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
    return check_hip(hipGetLastError(), "weight-only gemm kernel launch");
}

template <int FMT, int DT>
static int launch_wonly(hipStream_t stream, const uint8_t* x, int64_t ldx, const uint8_t* w, int64_t ldw, int M, int N, int K,
                        const float* scale, uint8_t* C, int64_t ldc) {
    // Up to 16 rows memory latency bounds it: 32 columns a workgroup where that leaves every CU with one, else 16.  With more
    // rows every workgroup's reading of all of x from the L2 does: as many columns as still give three CUs of four a workgroup
    // (64 rows, 14336 x 4096 with 16 / 32 / 64 columns: 72 / 45 / 32 us; 8192 x 8192: 69 / 41 / 53; 4096 x 14336: 60 / 68 / 88).
    const int64_t passes = M <= 64 ? 1 : (M + 63) / 64, enough = 3 * cu_count() / 4;
    if constexpr (DT != F8MI_FP32)
        if (M > 16 && passes * (N / 64) >= enough) return launch_wonly2<FMT, DT, 4>(stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
    if (M > 16 ? passes * (N / 32) >= enough : N > 32 * cu_count()) return launch_wonly2<FMT, DT, 2>(stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
    return launch_wonly2<FMT, DT, 1>(stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
}

template <int FMT>
static int wonly_dtype(int dtype, hipStream_t stream, const uint8_t* x, int64_t ldx, const uint8_t* w, int64_t ldw, int M, int N, int K,
                       const float* scale, uint8_t* C, int64_t ldc) {
    if (dtype == F8MI_BF16) return launch_wonly<FMT, F8MI_BF16>(stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
    if (dtype == F8MI_FP16) return launch_wonly<FMT, F8MI_FP16>(stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
    return launch_wonly<FMT, F8MI_FP32>(stream, x, ldx, w, ldw, M, N, K, scale, C, ldc);
}

template <int FMT>
static int dequant_dtype(int dtype, hipStream_t stream, const uint8_t* in, int64_t n, const float* scale, uint8_t* out) {
    const int64_t blocks = (n + 256 * 16 - 1) / (256 * 16);
    const dim3 g((unsigned)(blocks < 16384 ? blocks : 16384)), b(256);
    if (dtype == F8MI_BF16) hipLaunchKernelGGL((dequant_kernel<FMT, F8MI_BF16>), g, b, 0, stream, in, n, scale, out);
    else if (dtype == F8MI_FP16) hipLaunchKernelGGL((dequant_kernel<FMT, F8MI_FP16>), g, b, 0, stream, in, n, scale, out);
    else hipLaunchKernelGGL((dequant_kernel<FMT, F8MI_FP32>), g, b, 0, stream, in, n, scale, out);
    return check_hip(hipGetLastError(), "dequant kernel launch");
}

}  // namespace f8mi

using namespace f8mi;

extern "C" int f8mi_gemm_weight_only(const void* x, int64_t ldx, int dtype, const uint8_t* w, int fp8_fmt, int64_t ldw, int64_t m,
                                     int64_t n, int64_t k, const float* scale_dev, void* c, int64_t ldc, void* stream) {
    if (dtype < 0 || dtype > 2 || fp8_fmt < 0 || fp8_fmt > 1) { set_error("f8mi_gemm_weight_only: unknown dtype/format code"); return F8MI_ERR_INVALID_ARG; }
    if (m < 0 || n < 0 || k <= 0 || ldx < k || ldw < k || ldc < n) { set_error("f8mi_gemm_weight_only: bad shape m=%lld n=%lld k=%lld", (long long)m, (long long)n, (long long)k); return F8MI_ERR_INVALID_ARG; }
    if (m == 0 || n == 0) return F8MI_OK;
    if (m > 64 * 65535LL || n > 0x7fffff00LL || k > 0x7fffff00LL) { set_error("f8mi_gemm_weight_only: sizes past the grid's"); return F8MI_ERR_UNSUPPORTED; }
    if (!x || !w || !scale_dev || !c) { set_error("f8mi_gemm_weight_only: null pointer"); return F8MI_ERR_INVALID_ARG; }
    ProfScope prof(F8MI_K_GEMM, 2.0 * (double)m * (double)n * (double)k, (hipStream_t)stream);
    if (fp8_fmt == F8MI_E4M3FN) return wonly_dtype<F8MI_E4M3FN>(dtype, (hipStream_t)stream, (const uint8_t*)x, ldx, w, ldw, (int)m, (int)n, (int)k, scale_dev, (uint8_t*)c, ldc);
    return wonly_dtype<F8MI_E5M2>(dtype, (hipStream_t)stream, (const uint8_t*)x, ldx, w, ldw, (int)m, (int)n, (int)k, scale_dev, (uint8_t*)c, ldc);
}

extern "C" int f8mi_dequant(const uint8_t* in, int fp8_fmt, int64_t n, const float* scale_dev, int dtype, void* out, void* stream) {
    if (dtype < 0 || dtype > 2 || fp8_fmt < 0 || fp8_fmt > 1) { set_error("f8mi_dequant: unknown dtype/format code"); return F8MI_ERR_INVALID_ARG; }
    if (n < 0) { set_error("f8mi_dequant: bad size %lld", (long long)n); return F8MI_ERR_INVALID_ARG; }
    if (n == 0) return F8MI_OK;
    if (!in || !scale_dev || !out) { set_error("f8mi_dequant: null pointer"); return F8MI_ERR_INVALID_ARG; }
    ProfScope prof(F8MI_K_CAST, (double)n * (dtype == F8MI_FP32 ? 5 : 3), (hipStream_t)stream);
    if (fp8_fmt == F8MI_E4M3FN) return dequant_dtype<F8MI_E4M3FN>(dtype, (hipStream_t)stream, in, n, scale_dev, (uint8_t*)out);
    return dequant_dtype<F8MI_E5M2>(dtype, (hipStream_t)stream, in, n, scale_dev, (uint8_t*)out);
}
