// Implementation of the 16x16x128 LDS-DMA GEMM kernel, shared by the translation units that instantiate it
// for normal and transposed operands (f8mi_gemm_dma16*.hip).
#pragma once
#include "f8mi_gemm_util.h"

namespace f8mi {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int SLAB_BYTES = 256 * 128;   // one operand, one step
constexpr int HALF_BYTES = 256 * 64;    // one 64-deep unit of it
constexpr int NSLAB_A = 3, NSLAB_B = 2;

// TJ = 16-column tiles per wave: 8 -> 256 x 256 workgroup tiles; 7 -> 256 x 224 (see narrow_tiles_pay), operands as they are and rows of
// C at multiples of four bytes only.
template <int TJ>
struct LargeCfg {
    static constexpr int TILE_N = 32 * TJ;
    static constexpr int B_HALF = TILE_N * 64;  // one 64-deep unit of a slab of Bt
    static constexpr int B_SLAB = 2 * B_HALF;
    static constexpr int LDS = NSLAB_A * SLAB_BYTES + NSLAB_B * B_SLAB;
};

__device__ __forceinline__ void dma16b(const uint8_t* base, uint32_t voff, uint32_t lds_addr) {
    // M0 carries the LDS address; one wait state between the scalar write of M0 and its use
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" F8MI_DMA_CACHE_POLICY ::"v"(voff), "s"(base), "s"(lds_addr) : "memory");
}

// acc += first (16 rows x 128 k, format F1) * second^T (16 rows x 128 k, format F2); formats 0 = e4m3, 1 = e5m2.
// Written as an instruction so that the accumulator is an AGPR tuple updated in place: left to the
// register allocator, a quarter of the 64 accumulators ends up commuting between register files.
// The compiler does not know this is a matrix instruction: callers keep the required distance
// between the last one and the first read of an accumulator themselves.
template <int F1, int F2>
__device__ __forceinline__ void mfma16(v4f& acc, const v8i& first, const v8i& second) {
    asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:%3 blgp:%4" : "+a"(acc) : "v"(first), "v"(second), "n"(F1), "n"(F2));
}
// acc = first * second^T: the first step of a tile starts from the constant 0 instead of zeroed
// registers (a register written by an ordinary vector instruction must not be read by a matrix
// instruction right away, and nothing here would keep the compiler from placing the two back to back).
template <int F1, int F2>
__device__ __forceinline__ void mfma16_first(v4f& acc, const v8i& first, const v8i& second) {
    asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0 cbsz:%3 blgp:%4" : "=a"(acc) : "v"(first), "v"(second), "n"(F1), "n"(F2));
}

// One accumulator register into a vector register, as an instruction of its own: it stays where it is written
// relative to the MFMAs (also volatile asm).  Left to the compiler, which takes the MFMAs for ordinary
// instructions, the copy may be placed right behind the MFMA that produces the value, where it reads the old one.
__device__ __forceinline__ float acc_read(float a) {
    float v;
    asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(a));
    return v;
}

// The epilogue: scales the 8 x 8 (TJ x 8) tiles of 16 x 16 accumulators, adds the bias, converts and writes C.
// acc[tj][ti] as left by MFMA(first = Bt rows, second = A rows): lane holds row ti*16 + lane%16
// and the four columns tj*16 + 4*(lane/16) + e of its wave's 128 x 128 quarter.
//
// 16-bit outputs go straight from the registers, one `piece` = one store instruction at a time, so that the
// kernel can slot the pieces of a finished row of tiles between the MFMAs of the next row in its last step.
// A lane holds 4 neighbouring columns of a row (8 bytes) of each accumulator tile; v_permlane16_swap between the
// tiles tj = 2p and 2p + 1 trades the odd 16-lane rows of the first for the even ones of the second, after which
// every lane holds 8 neighbouring columns (lq even: columns 4 lq .. 4 lq + 7 of tile 2p; lq odd: columns
// 4 (lq - 1) .. + 7 of tile 2p + 1) and one 16-byte store per lane writes 64 contiguous bytes of 16 rows.
// (Staging the tile through LDS for 256-byte row segments takes the same time and needs the slabs to be free.)
// A piece of an fp32 C is a lane's own four columns of either tile, two 16-byte stores (us, all of the tile written
// behind the last MFMA / piece by piece: 4096 x 4096 over 4096 54.8 / 51.4, 8192 x 4096 over 1024 47.9 / 40.7, 8192 x 14336 over 4096 404 / 358,
// 4099 x 11007 over 4224 186 / 150).
// ODD_ROWS: rows of C start at odd multiples of two bytes too (see ShiftedRows); a piece is then stored behind the next one.
template <int C_DT, bool ODD_ROWS, int TJ, bool BIAS_AFTER>
struct Epilogue16 {
    int M, N, c_vec_ok, lq, row0, col0, wcol0;
    bool whole, interior;  // the 256 x 256 tile lies inside C; and its rows take 16-byte stores as they are (the same for every lane)
    uint16_t* base;  // of the lane's first piece: a piece's address is this plus an offset that is the same for every lane
    float* base32;   // the same of an fp32 C
    float inv;
    int64_t ldc;
    void* C;
    const void* bias;
    int bias_fp32;
    ShiftedRows rows_shifted;
    float bv[TJ][4];

    __device__ __forceinline__ Epilogue16(int m0, int n0, int M_, int N_, float inv_, void* C_, int64_t ldc_, const void* bias_,
                                          int bias_fp32_, int c_vec_ok_)
        : M(M_), N(N_), c_vec_ok(c_vec_ok_), inv(inv_), ldc(ldc_), C(C_), bias(bias_), bias_fp32(bias_fp32_),
          rows_shifted(C_, ldc_, m0 + (int)(threadIdx.x >> 7) * 128 + (int)(threadIdx.x & 15)) {
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        lq = lane >> 4;
        wcol0 = n0 + (wave & 1) * (16 * TJ);
        row0 = m0 + (wave >> 1) * 128 + (lane & 15);
        col0 = wcol0 + (lq & 1) * 16 + (lq >> 1) * 8;  // of the lane's 8 columns in the first pair of tiles
        whole = m0 + 256 <= M && n0 + 32 * TJ <= N;
        interior = c_vec_ok && whole;
        base = (uint16_t*)C + (int64_t)row0 * ldc + col0;
        base32 = (float*)C + (int64_t)row0 * ldc + wcol0 + 4 * lq;
    }

    __device__ __forceinline__ void load_bias_row() {
        if constexpr (c_is_fp32(C_DT)) load_bias_tiles<F8MI_FP32, TJ>(bv, bias, wcol0 + 4 * lq, N);
        else if constexpr (BIAS_AFTER) load_rounded_bias_tiles<C_DT, TJ>(bv, bias, bias_fp32, wcol0 + 4 * lq, N);
        else load_bias_tiles<C_DT, TJ>(bv, bias, wcol0 + 4 * lq, N);
    }

    __device__ __forceinline__ void store_held(int ti, int tp) {
        uint16_t* dst = base + ((int64_t)(ti * 16) * ldc + tp * 32);
        if (whole) rows_shifted.store(dst, true, tp == 0, tp == 3, 0, 0, M, N);
        else rows_shifted.store(dst, false, tp == 0, tp == 3, row0 + ti * 16, col0 + tp * 32, M, N);
    }
    __device__ __forceinline__ void finish() {  // behind the last piece
        if constexpr (ODD_ROWS) store_held(7, 3);
    }

    // rows ti*16 .. +15, columns tp*32 .. +31 of the wave's quarter; every lane must call it; pieces of a row of
    // tiles from left to right, rows from the top
    __device__ __forceinline__ void piece(v4f (&acc)[TJ][8], int ti, int tp) {
        const int te = 2 * tp, to = 2 * tp + 1;
        float e[4], o[4];
#pragma unroll
        for (int r = 0; r < 4; r++) e[r] = acc_read(acc[te][ti][r]);
#pragma unroll
        for (int r = 0; r < 4; r++) o[r] = acc_read(acc[to][ti][r]);
        if constexpr (c_is_fp32(C_DT)) {
            const int r = row0 + ti * 16, c = wcol0 + te * 16 + 4 * lq;
            float* dst = base32 + ((int64_t)(ti * 16) * ldc + tp * 32);
            store_fp32x4(dst, finish4<C_DT, BIAS_AFTER>(e, inv, bv[te]), interior, c_vec_ok, r, c, M, N);
            store_fp32x4(dst + 16, finish4<C_DT, BIAS_AFTER>(o, inv, bv[to]), interior, c_vec_ok, r, c + 16, M, N);
            return;
        }
        const uint32_t x0 = finish2<C_DT, BIAS_AFTER>(e[0], e[1], inv, bv[te][0], bv[te][1]);
        const uint32_t x1 = finish2<C_DT, BIAS_AFTER>(e[2], e[3], inv, bv[te][2], bv[te][3]);
        const uint32_t y0 = finish2<C_DT, BIAS_AFTER>(o[0], o[1], inv, bv[to][0], bv[to][1]);
        const uint32_t y1 = finish2<C_DT, BIAS_AFTER>(o[2], o[3], inv, bv[to][2], bv[to][3]);
        const auto s0 = __builtin_amdgcn_permlane16_swap(x0, y0, false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(x1, y1, false, false);
        if constexpr (ODD_ROWS) {
            if (tp > 0) store_held(ti, tp - 1);
            else if (ti > 0) store_held(ti - 1, 3);
            rows_shifted.hold(make_uint4(s0[0], s1[0], s0[1], s1[1]));
            return;
        }
        const int row = row0 + ti * 16, col = col0 + tp * 32;
        // A tile inside C checks nothing: one scalar branch instead of the per-lane comparisons, the address one vector
        // instruction (the lane's base plus an offset that is the same for all lanes), and the element-wise tail -- 60 of
        // a piece's 90 instructions -- out of the way.  The last step of a tile is bound by the vector ALU, not by the
        // matrix core (an MFMA keeps the ALU from issuing for about 16 of its 32 cycles, and what follows costs 4 - 5
        // cycles per instruction: 165 cycles per pair of MFMAs with a piece behind it, measured on one wave), so every
        // instruction less in a piece is time: 16384 x 8192 x K products 0.8 / 1.0 / 2.0 % faster at K = 8192 / 4096 / 2048.
        if (__builtin_expect(interior, 1)) {
            store16_any(base + ((int64_t)(ti * 16) * ldc + tp * 32), make_uint4(s0[0], s1[0], s0[1], s1[1]));
            return;
        }
        if (row < M && col < N) {
            uint16_t* dst = (uint16_t*)C + (int64_t)row * ldc + col;
            if (c_vec_ok && col + 8 <= N) {
                store16_any(dst, make_uint4(s0[0], s1[0], s0[1], s1[1]));
            } else {
                const uint32_t w[4] = {s0[0], s1[0], s0[1], s1[1]};
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (col + i < N) dst[i] = (uint16_t)((w[i >> 1] >> (16 * (i & 1))) & 0xffffu);
            }
        }
    }

    // the last column of tiles of an odd number, rows ti*16 .. +15: a lane's own 4 columns, 8 bytes
    __device__ __forceinline__ void piece_last(v4f (&acc)[TJ][8], int ti) {
        constexpr int tj = TJ - 1;
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; r++) e[r] = acc_read(acc[tj][ti][r]);
        if constexpr (c_is_fp32(C_DT)) {
            store_fp32x4(base32 + ((int64_t)(ti * 16) * ldc + tj * 16), finish4<C_DT, BIAS_AFTER>(e, inv, bv[tj]), interior, c_vec_ok, row0 + ti * 16,
                         wcol0 + tj * 16 + 4 * lq, M, N);
            return;
        }
        const uint32_t x0 = finish2<C_DT, BIAS_AFTER>(e[0], e[1], inv, bv[tj][0], bv[tj][1]);
        const uint32_t x1 = finish2<C_DT, BIAS_AFTER>(e[2], e[3], inv, bv[tj][2], bv[tj][3]);
        const int row = row0 + ti * 16, col = wcol0 + tj * 16 + 4 * lq;
        uint16_t* dst = (uint16_t*)C + (int64_t)row * ldc + col;
        if (__builtin_expect(interior, 1)) {
            store8_any(dst, x0, x1);
            return;
        }
        if (row < M && col < N) {
            if (c_vec_ok && col + 4 <= N) {
                store8_any(dst, x0, x1);
            } else {
                const uint32_t w[2] = {x0, x1};
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (col + i < N) dst[i] = (uint16_t)((w[i >> 1] >> (16 * (i & 1))) & 0xffffu);
            }
        }
    }
};

// ODD (from the host): the number of steps K/128 is odd.
// A_TR / B_TR: the operand is given "transposed": its memory holds the matrix [contraction][rows] (the layout
// in which another GEMM contracts over `rows`), a slab is 128 contraction rows x 256 row-bytes, and fragments
// are built with ds_read_b64_tr_b8.  For such an operand lda / ldb is the byte distance between contraction
// rows (64 when k-blocked over `rows`, the row stride when row-major) and a_unit / b_unit the distance between
// blocks of 64 rows (contraction length * 64 when k-blocked, 64 when row-major).
// Workgroup `lid` of the `npid` that compute this product.
template <int AF, int BF, int C_DT, bool ODD, bool A_TR, bool B_TR, bool ODD_ROWS, int TJ, bool BIAS_AFTER = false>
__device__ __forceinline__ void gemm_dma16_tile(
    int lid, const int npid, const uint8_t* __restrict__ A, int64_t lda, int64_t a_unit, const uint8_t* __restrict__ Bt, int64_t ldb, int64_t b_unit,
    int M, int N, int K, const float* __restrict__ sa_dev, const float* __restrict__ sb_dev, void* __restrict__ C,
    int64_t ldc, const void* __restrict__ bias, int tiles_m, int tiles_n, int c_vec_ok, int bias_fp32 = 0) {
    static_assert(TJ == 8 || (TJ == 7 && !A_TR && !B_TR && !ODD_ROWS), "narrower tiles: operands as they are");
    using Cfg = LargeCfg<TJ>;
    extern __shared__ __align__(16) uint8_t smem[];
    // lda / ldb: bytes from one operand row to the next; a_unit / b_unit: bytes from one 64-deep unit
    // to the next.  Row-major operands: (row stride, 64); k-blocked [K/64][rows][64]: (64, rows*64).

    // ---- which tile (same walk as the other kernels)
#if F8MI_WALK_XCD_CHUNK == 0
    lid = xcd_contiguous_id(lid, npid);
#else
    {   // measurement builds only: chunks of F8MI_WALK_XCD_CHUNK tile ids dealt round-robin to the XCDs
        const int full = npid - npid % (NUM_XCD * F8MI_WALK_XCD_CHUNK);
        if (lid < full) {
            const int x = lid % NUM_XCD, j = lid / NUM_XCD;
            lid = ((j / F8MI_WALK_XCD_CHUNK) * NUM_XCD + x) * F8MI_WALK_XCD_CHUNK + (j % F8MI_WALK_XCD_CHUNK);
        }
    }
#endif
    // The walk sweeps along the longer side of the tile grid in bands GROUP tiles wide, so that an XCD's 32
    // workgroups hold a 4 x 8 (or 8 x 4) patch of neighbouring tiles; sweeping along the shorter side instead
    // cost 1 - 3 % on the shapes where the sides differ most (measured both ways on all twelve benchmark GEMMs).
    // Per 128-deep step such a patch pulls 4 + 8 operand panels through the XCD's L2 for 32 tiles, the least that 32
    // tiles in step allow; bytes fetched past the L2 and GEMM rate by band width, same box, benchmark step: 1 tile
    // 14.2 GB per launch / 2982 TFLOP/s, 2 tiles 7.8 / 3190, 4 tiles 5.2 / 3250, 8 tiles 5.2 / 3259, 16 tiles - / 3187.
    constexpr int GROUP = F8MI_WALK_GROUP;
    int tm, tn;
    if ((tiles_m > tiles_n) != (F8MI_WALK_SHORT_SIDE != 0)) {
        const int width = GROUP * tiles_m;
        const int first_n = (lid / width) * GROUP;
        const int gsz = min(tiles_n - first_n, GROUP);
        tn = first_n + (lid % width) % gsz;
        tm = (lid % width) / gsz;
    } else {
        const int width = GROUP * tiles_n;
        const int first_m = (lid / width) * GROUP;
        const int gsz = min(tiles_m - first_m, GROUP);
        tm = first_m + (lid % width) % gsz;
        tn = (lid % width) / gsz;
    }
    const int m0 = tm * BM, n0 = tn * Cfg::TILE_N;
    // 1 / (sa * sb) for the epilogue, fetched now and kept in a scalar register: loaded after the main loop, the two
    // scales were a memory round trip with nothing to hide it
    const float inv = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(
        int, __fdiv_rn(1.0f, *sa_dev) * __fdiv_rn(1.0f, *sb_dev))));

    const int t = threadIdx.x;
    const int lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // ---- DMA addressing.
    // Normal operand: instruction j = wave*4 + i of a slab half covers tile rows 16j .. 16j+15; lane l fetches
    // row 16j + l/4, 16-byte piece (l%4) ^ (l/32) -- the swizzle, applied on the global side: rows 8..15 of every
    // sixteen hold their pieces in the order 1, 0, 3, 2.
    // A 16-byte LDS read serves the lanes 0-3, 12-15, 20-23, 24-27 together, then 4-7, 8-11, 16-19, 28-31, then
    // the same of the upper 32 (found by timing address patterns); with this swizzle each such group of a
    // fragment read covers all 64 banks.  (piece ^ (row/4) % 4, the usual choice, made every read take twice
    // its cycles: SQ_LDS_BANK_CONFLICT was half of SQ_LDS_IDX_ACTIVE.)
    // Transposed operand: instruction j = wave*8 + d covers contraction rows 4j .. 4j+3 of the slab, 256 bytes
    // (16 slots) each; lane l fetches row 4j + l/16, the slot that belongs at position l%16: (l%16) ^ f(row).
    const uint32_t lds_u32 = (uint32_t)(uintptr_t)smem;
    uint32_t a_voff[A_TR ? 8 : 4], b_voff[B_TR ? 8 : TJ == 8 ? 4 : TJ];
    const uint8_t* a_ptr;  // first byte of the next step to be fetched
    const uint8_t* b_ptr;
    int64_t a_step, b_step;  // bytes from one step's data to the next
    if constexpr (A_TR) {
#pragma unroll
        for (int d = 0; d < 8; d++) {
            const int rowl = 4 * (wave * 8 + d) + (lane >> 4);
            const int c = (lane & 15) ^ tr_swizzle(rowl);
            const int blk = min(m0 / 64 + (c >> 2), M / 64 - 1) - m0 / 64;  // blocks past the edge re-read the last one
            a_voff[d] = (uint32_t)(rowl * lda + blk * a_unit) + (c & 3) * 16;
        }
        a_ptr = A + (int64_t)(m0 / 64) * a_unit;
        a_step = 128 * lda;
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = (wave * 4 + i) * 16 + (lane >> 2);
            a_voff[i] = (uint32_t)(min(r, M - 1 - m0) * lda) + (((lane & 3) ^ (lane >> 5)) << 4);  // rows past the edge re-read the last row
        }
        a_ptr = A + (int64_t)m0 * lda;
        a_step = 2 * a_unit;
    }
    if constexpr (B_TR) {
#pragma unroll
        for (int d = 0; d < 8; d++) {
            const int rowl = 4 * (wave * 8 + d) + (lane >> 4);
            const int c = (lane & 15) ^ tr_swizzle(rowl);
            const int blk = min(n0 / 64 + (c >> 2), N / 64 - 1) - n0 / 64;
            b_voff[d] = (uint32_t)(rowl * ldb + blk * b_unit) + (c & 3) * 16;
        }
        b_ptr = Bt + (int64_t)(n0 / 64) * b_unit;
        b_step = 128 * ldb;
    } else {
        // 256 rows: as for A; fewer: wave w takes TJ of the 2 TJ instructions of the half w / 2
#pragma unroll
        for (int i = 0; i < (TJ == 8 ? 4 : TJ); i++) {
            const int r = (TJ == 8 ? wave * 4 + i : (wave & 1) * TJ + i) * 16 + (lane >> 2);
            b_voff[i] = (uint32_t)(min(r, N - 1 - n0) * ldb) + (((lane & 3) ^ (lane >> 5)) << 4);
        }
        b_ptr = Bt + (int64_t)n0 * ldb + (TJ == 8 ? 0 : (wave >> 1) * b_unit);
        b_step = 2 * b_unit;
    }
    uint32_t a_dst = 0, b_dst = 0;  // LDS address of the slabs being refilled
    // DMA d = 0..7 of this wave's share of a slab
    auto issue_a = [&](int d) __attribute__((always_inline)) {
        if constexpr (A_TR) dma16b(a_ptr, a_voff[d], a_dst + (wave * 8 + d) * 1024);
        else dma16b(d < 4 ? a_ptr : a_ptr + a_unit, a_voff[d & 3], a_dst + wave * 4096 + (d >> 2) * HALF_BYTES + (d & 3) * 1024);
        if (d == 7) a_ptr += a_step;
    };
    auto issue_b = [&](int d) __attribute__((always_inline)) {
        if constexpr (B_TR) dma16b(b_ptr, b_voff[d], b_dst + (wave * 8 + d) * 1024);
        else if constexpr (TJ == 8) dma16b(d < 4 ? b_ptr : b_ptr + b_unit, b_voff[d & 3], b_dst + wave * 4096 + (d >> 2) * HALF_BYTES + (d & 3) * 1024);
        else dma16b(b_ptr, b_voff[d], b_dst + (wave * TJ + d) * 1024);
        if (d == TJ - 1) b_ptr += b_step;
    };

    // ---- fragment addressing.
    // Normal operand: lane -> tile row lane % 16, k quarter lane / 16 (32 bytes: half q/2, pieces 2(q%2), 2(q%2)+1).
    // Transposed operand: lane j of a 16-lane group q addresses contraction row 32q + 8t + j/2 (t-th read),
    // byte column tile*16 + 8*(j%2) of the wave's 128 columns, through the slot swizzle.
    const int frow = lane & 15, fq = lane >> 4;
    const int fsw = (frow >> 3) & 1;
    const int f_off0 = (fq >> 1) * HALF_BYTES + frow * 64 + ((((fq & 1) * 2 + 0) ^ fsw) << 4);
    const int f_off1 = (fq >> 1) * HALF_BYTES + frow * 64 + ((((fq & 1) * 2 + 1) ^ fsw) << 4);
    const int tr_f = tr_swizzle(32 * fq + (frow >> 1));  // the same for all four reads of a lane
    int a_tr_off[A_TR ? 8 : 1], b_tr_off[B_TR ? 8 : 1];
    if constexpr (A_TR) {
        const int base = (32 * fq + (frow >> 1)) * 256 + 128 * (wm ^ (tr_f >> 3)) + 8 * (frow & 1);
#pragma unroll
        for (int x = 0; x < 8; x++) a_tr_off[x] = base + ((x ^ (tr_f & 7)) << 4);
    }
    if constexpr (B_TR) {
        const int base = (32 * fq + (frow >> 1)) * 256 + 128 * (wn ^ (tr_f >> 3)) + 8 * (frow & 1);
#pragma unroll
        for (int x = 0; x < 8; x++) b_tr_off[x] = base + ((x ^ (tr_f & 7)) << 4);
    }
    const int a_frag_base = (wm * 128) * 64;
    const int b_frag_base = (wn * (16 * TJ)) * 64 + (fq >> 1) * (Cfg::B_HALF - HALF_BYTES);
    auto frag_a = [&](const uint8_t* slab, int ti) __attribute__((always_inline)) {
        if constexpr (A_TR) {
            return read_frag_tr(slab + a_tr_off[ti]);
        } else {
            const uint8_t* p = slab + a_frag_base + ti * 16 * 64;
            return read_frag(p + f_off0, p + f_off1);
        }
    };
    auto frag_b = [&](const uint8_t* slab, int tj) __attribute__((always_inline)) {
        if constexpr (B_TR) {
            return read_frag_tr(slab + b_tr_off[tj]);
        } else {
            const uint8_t* p = slab + b_frag_base + tj * 16 * 64;
            return read_frag(p + f_off0, p + f_off1);
        }
    };

    v4f acc[TJ][8];  // first written by step 0

    v8i fb[2][TJ];  // [step parity][n tile]
    v8i fa[2];     // rolling: group ti multiplies fa[ti & 1] while fa[(ti + 1) & 1] is being fetched

    // ---- prologue: steps 0 and 1 (A into slabs 0, 1; Bt into slabs 3, 4), wait for step 0,
    // first fragments; a second barrier before step 0 refills the Bt slab just read.
#pragma unroll
    for (int s = 0; s < 2; s++) {
        a_dst = lds_u32 + s * SLAB_BYTES;
        b_dst = lds_u32 + NSLAB_A * SLAB_BYTES + s * Cfg::B_SLAB;
#pragma unroll
        for (int d = 0; d < 8; d++) issue_a(d);
#pragma unroll
        for (int d = 0; d < TJ; d++) issue_b(d);
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 + TJ) : "memory");
    lds_barrier();
#pragma unroll
    for (int x = 0; x < TJ; x++) fb[0][x] = frag_b(smem + NSLAB_A * SLAB_BYTES, x);
    fa[0] = frag_a(smem, 0);
    lds_barrier();

    // One step t.  P: parity of t.  MODE 0: steps t+1 and t+2 exist (refills the slabs freed at this
    // step's start with step t+2); 1: last but one (nothing left to fetch); 2: last step; 3: step 0 (as 0,
    // and the accumulators start from zero).
    int a_slab = 0;  // slab of A of this step; step t+2 goes to the slab before it in the rotation
    Epilogue16<C_DT, ODD_ROWS, TJ, BIAS_AFTER> epi(m0, n0, M, N, inv, C, ldc, bias, bias_fp32, c_vec_ok);
    auto step = [&](auto parity, auto mode) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value;
        constexpr bool FIRST = decltype(mode)::value == 3;
        constexpr int MODE = FIRST ? 0 : decltype(mode)::value;
        const int a_next = a_slab + 1 == NSLAB_A ? 0 : a_slab + 1;
        const int a_free = a_next + 1 == NSLAB_A ? 0 : a_next + 1;  // held step t-1
        const uint8_t* a_cur = smem + a_slab * SLAB_BYTES;
        const uint8_t* a_nxt = smem + a_next * SLAB_BYTES;
        const uint8_t* b_nxt = smem + NSLAB_A * SLAB_BYTES + (P ^ 1) * Cfg::B_SLAB;
        if (MODE == 0) {
            a_dst = lds_u32 + a_free * SLAB_BYTES;
            b_dst = lds_u32 + NSLAB_A * SLAB_BYTES + P * Cfg::B_SLAB;  // Bt of this step: already in registers
        }
        // Everything that is not an MFMA sits in a fixed slot between two MFMAs (each keeps the matrix
        // core busy for 32 cycles): one fragment (two 16-byte LDS reads) or one DMA at a time.
        // The last step has neither; there the finished row of accumulator tiles (ti - 1: its last MFMA was issued
        // eight MFMAs before the first read) is scaled, converted and stored under the MFMAs of row ti.
        if (MODE == 2) epi.load_bias_row();
#pragma unroll
        for (int ti = 0; ti < 8; ti++) {
            if (ti == 6 && MODE < 2) {
                // this wave's DMAs of step t+1 have landed (the 12 of step t+2 issued so far may be in flight) ...
                if (MODE == 0) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                asm volatile("s_barrier" ::: "memory");  // ... and so have everybody's; no LDS hazard here, so no wait on LDS reads
            }
#pragma unroll
            for (int tj = 0; tj < TJ; tj++) {
                if (tj == 0 && ti < 7) fa[(ti + 1) & 1] = frag_a(a_cur, ti + 1);
                if (tj == 0 && ti == 7 && MODE < 2) fa[0] = frag_a(a_nxt, 0);
                if constexpr (TJ == 8) {
                    if (MODE < 2 && ti >= 6 && (tj & 1) == 1) fb[P ^ 1][(ti - 6) * 4 + (tj >> 1)] = frag_b(b_nxt, (ti - 6) * 4 + (tj >> 1));
                } else {  // four of the seven in the last but one row, three in the last
                    if (MODE < 2 && ti == 6 && (tj == 1 || tj == 3 || tj >= 5)) fb[P ^ 1][tj == 6 ? 3 : tj >> 1] = frag_b(b_nxt, tj == 6 ? 3 : tj >> 1);
                    if (MODE < 2 && ti == 7 && (tj & 1) == 1) fb[P ^ 1][4 + (tj >> 1)] = frag_b(b_nxt, 4 + (tj >> 1));
                }
                if (FIRST) mfma16_first<BF, AF>(acc[tj][ti], fb[P][tj], fa[ti & 1]);
                else mfma16<BF, AF>(acc[tj][ti], fb[P][tj], fa[ti & 1]);
                F8MI_SCHED_FENCE();
                // (seven tiles: a place later, and the last one in the row after, for the same distance from the MFMA that wrote it)
                if (MODE == 2 && ti >= 1 && (TJ == 8 ? (tj & 1) == 1 : tj >= 2 && (tj & 1) == 0)) {
                    epi.piece(acc, ti - 1, TJ == 8 ? tj >> 1 : (tj >> 1) - 1);
                    F8MI_SCHED_FENCE();
                }
                if constexpr (TJ == 7) {
                    if (MODE == 2 && ti >= 2 && tj == 1) {
                        epi.piece_last(acc, ti - 2);
                        F8MI_SCHED_FENCE();
                    }
                }
                if (MODE == 0 && (tj & 3) == 0) {
                    // 16 DMAs over the 64 MFMAs, one after every fourth: A slab first, then Bt.  (Packed into
                    // the first half of the step they cost 3 % more time: the four waves share one load unit.)
                    const int d = ti * 2 + (tj >> 2);
                    if (d < 8) issue_a(d);
                    else if (d - 8 < TJ) issue_b(d - 8);
                    F8MI_SCHED_FENCE();
                }
            }
        }
        if (MODE < 2) lds_barrier();  // step boundary: everybody is done with A of step t and has Bt of step t+1 in registers
        a_slab = a_next;
    };

    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    constexpr std::integral_constant<int, 2> c2{};

    constexpr std::integral_constant<int, 3> c3{};
    const int n_steady = K / 128 - 2;  // steps that fetch: >= 1 (host); ODD <=> odd
    step(c0, c3);
    if constexpr (ODD) {
        for (int s = 1; s < n_steady; s += 2) {
            step(c1, c0);
            step(c0, c0);
        }
        step(c1, c1);
        step(c0, c2);
    } else {
        step(c1, c0);
        for (int s = 2; s < n_steady; s += 2) {
            step(c0, c0);
            step(c1, c0);
        }
        step(c0, c1);
        step(c1, c2);
    }
    // the last MFMAs are still in the pipeline (8 passes): keep the accumulator reads away from them.  (No DMA is
    // outstanding: the last but one step waited for all of them.)
    asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int tp = 0; tp < TJ / 2; tp++) epi.piece(acc, 7, tp);
    if constexpr (TJ == 7) {
        epi.piece_last(acc, 6);
        epi.piece_last(acc, 7);
    }
    epi.finish();
}

template <int AF, int BF, int C_DT, bool ODD, bool A_TR, bool B_TR, bool ODD_ROWS, int TJ>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_nt_dma16_kernel(
    const uint8_t* __restrict__ A, int64_t lda, int64_t a_unit, const uint8_t* __restrict__ Bt, int64_t ldb, int64_t b_unit,
    int M, int N, int K, const float* __restrict__ sa_dev, const float* __restrict__ sb_dev, void* __restrict__ C,
    int64_t ldc, const void* __restrict__ bias, int tiles_m, int tiles_n, int c_vec_ok) {
    gemm_dma16_tile<AF, BF, C_DT, ODD, A_TR, B_TR, ODD_ROWS, TJ>(blockIdx.x, gridDim.x, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa_dev, sb_dev, C,
                                                                 ldc, bias, tiles_m, tiles_n, c_vec_ok);
}

template <int AF, int BF, int C_DT, bool ODD, bool A_TR, bool B_TR, bool ODD_ROWS, int TJ>
static int launch16_4(dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit, const uint8_t* Bt, int64_t ldb,
                      int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C, int64_t ldc,
                      const void* bias, int tiles_m, int tiles_n, int c_vec_ok) {
    static std::atomic<uint64_t> lds_allowed{0};
    auto kern = gemm_nt_dma16_kernel<AF, BF, C_DT, ODD, A_TR, B_TR, ODD_ROWS, TJ>;
    if (int rc = allow_big_lds(kern, LargeCfg<TJ>::LDS, lds_allowed)) return rc;
    hipLaunchKernelGGL(kern, g, dim3(GEMM_THREADS), LargeCfg<TJ>::LDS, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C,
                       ldc, bias, tiles_m, tiles_n, c_vec_ok);
    return check_hip(hipGetLastError(), "gemm (LDS-DMA, 16x16x128) kernel launch");
}

template <int AF, int BF, int C_DT, bool A_TR, bool B_TR, bool ODD_ROWS, int TJ>
static int launch16_3(dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit, const uint8_t* Bt, int64_t ldb,
                      int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C, int64_t ldc,
                      const void* bias, int tiles_m, int tiles_n, int c_vec_ok) {
    if ((K / 128) & 1) return launch16_4<AF, BF, C_DT, true, A_TR, B_TR, ODD_ROWS, TJ>(g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
    return launch16_4<AF, BF, C_DT, false, A_TR, B_TR, ODD_ROWS, TJ>(g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
}

template <int AF, int BF, bool A_TR, bool B_TR, bool ODD_ROWS, int TJ>
static int launch16_2(int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit, const uint8_t* Bt,
                      int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C, int64_t ldc,
                      const void* bias, int tiles_m, int tiles_n, int c_vec_ok) {
    if (c_dtype == F8MI_BF16) return launch16_3<AF, BF, F8MI_BF16, A_TR, B_TR, ODD_ROWS, TJ>(g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
    if (c_dtype == F8MI_FP16) return launch16_3<AF, BF, F8MI_FP16, A_TR, B_TR, ODD_ROWS, TJ>(g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
    if constexpr (ODD_ROWS) { set_error("gemm: fp32 rows are never at odd multiples of two bytes"); return F8MI_ERR_INVALID_ARG; }
    else return launch16_3<AF, BF, F8MI_FP32, A_TR, B_TR, false, TJ>(g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
}

template <bool A_TR, bool B_TR, bool ODD_ROWS = false, int TJ = 8>
static int launch_gemm_dma16_t(int a_fmt, int b_fmt, int c_dtype, dim3 g, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                      const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb,
                      void* C, int64_t ldc, const void* bias, int tiles_m, int tiles_n, int c_vec_ok) {
    if (a_fmt == F8MI_E4M3FN && b_fmt == F8MI_E4M3FN) return launch16_2<0, 0, A_TR, B_TR, ODD_ROWS, TJ>(c_dtype, g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
    if (a_fmt == F8MI_E5M2 && b_fmt == F8MI_E4M3FN) return launch16_2<1, 0, A_TR, B_TR, ODD_ROWS, TJ>(c_dtype, g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
    if (a_fmt == F8MI_E4M3FN && b_fmt == F8MI_E5M2) return launch16_2<0, 1, A_TR, B_TR, ODD_ROWS, TJ>(c_dtype, g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
    return launch16_2<1, 1, A_TR, B_TR, ODD_ROWS, TJ>(c_dtype, g, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok);
}

}  // namespace f8mi
