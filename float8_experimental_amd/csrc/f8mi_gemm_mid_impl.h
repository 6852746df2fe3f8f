// K3 for outputs of few 256 x 256 tiles: the same 16x16x128 MFMA, LDS-DMA and LDS layout as
// f8mi_gemm_dma16_impl.h on tiles of 128 rows, so that two or four times as many workgroups share the CUs.
//
// The large-tile kernel is built for the regime where every CU has tiles queued: one workgroup owns a CU
// (160 KB of LDS, 512 registers per lane) and walks all of k in 1.1 us steps -- 70 us for k = 8192 however
// few tiles there are.  With 512 rows and 8192 columns that is 64 workgroups on 256 CUs.  Here a workgroup
// (4 waves as 2 x 2) takes a tile of 128 x 128 (64 x 64 per wave, 16 accumulator tiles, five LDS stages of
// (128 + 128 rows) x 128 k) or 128 x 256 (64 x 128 per wave, three stages of (128 + 256 rows) x 128 k): 256
// workgroups for that output with the former, and one round of workgroups instead of two for outputs of 65 to 128
// large tiles with the latter.
//
// One wave per SIMD has nobody to hide its waits behind, so a step waits for nothing that is not long done: the
// fragments of the next step are read into a second set of registers while this step's are multiplied, two 16-byte
// reads after every second MFMA and a DMA after the others (an MFMA leaves room for one of the two), the DMAs
// into the stage whose fragments all waves already hold; one barrier per step.  Reading a step's fragments at its
// start instead, with a second barrier at its end, left the matrix cores idle for half of the step: 2048 x 4096 over
// k = 4096: 35.8 -> 30.1 us (128 x 256 tiles), 1024 x 4096 over 8192: 39.2 -> 31.3 (128 x 128), 512 x 1024 over 1024:
// 8.5 -> 6.6.  What is left: 0.70 us a step of 128 x 256 tiles, of which the MFMAs alone need 0.55 at the clock the
// power cap leaves them (measured without the DMAs), and 8 us a launch for the first DMAs, the stores of C and the launch.
//
// A_TR / B_TR: the operand's memory holds [contraction][rows] (f8mi_gemm_dma16_impl.h has the addressing): a stage then keeps
// 128 contraction rows of 128 or 256 bytes of it and fragments are built with ds_read_b64_tr_b8.
//
// A wave's accumulation order over k is that of the large-tile kernels (128-deep steps in sequence, the same
// 32 contraction bytes per lane), so the results are the same bits.
// Host side guarantees: K % 128 == 0, K >= 128, 16-byte aligned operands and strides.
#pragma once
#include "f8mi_gemm_util.h"

namespace f8mi {

typedef float v4f_m __attribute__((ext_vector_type(4)));

constexpr int MID_TILE_M = 128;
constexpr int MID_A_UNIT = MID_TILE_M * 64;  // A, one 64-deep unit of a stage: 8 KB

// TJ = 16-column tiles per wave: 4 -> 128 x 128 workgroup tiles, five stages of 32 KB;
//                                8 -> 128 x 256, three stages of 48 KB.
template <int TJ>
struct MidCfg {
    static constexpr int TILE_N = 32 * TJ;
    static constexpr int B_UNIT = TILE_N * 64;
    static constexpr int STAGE = 2 * MID_A_UNIT + 2 * B_UNIT;
    static constexpr int NSTAGE = TJ == 4 ? 5 : 3;
    static constexpr int LDS = NSTAGE * STAGE;  // 160 KB / 144 KB
    static constexpr int BI = TJ / 2;           // Bt row groups (16 rows) per wave and unit
    static constexpr int NDMA = 4 + 2 * BI;     // DMAs per wave and step
};

__device__ __forceinline__ void dma_mid(const uint8_t* base, uint32_t voff, uint32_t lds_addr) {
    // M0 carries the LDS address; one wait state between the scalar write of M0 and its use
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base), "s"(lds_addr) : "memory");
}

// A float through the scalar cache (the address is the same for every lane).
__device__ __forceinline__ float load_scalar(const float* p) { return *(const __attribute__((address_space(4))) float*)p; }

// Waits until at most N of this wave's DMAs are in flight and none of its LDS reads, then for the whole workgroup.
template <int N>
__device__ __forceinline__ void mid_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// f(k) of the slot swizzle of a transposed operand: the 16-byte slot c of contraction row k sits at slot c ^ f(k).  The 16 rows
// that 32 lanes of a transpose read touch (8t .. 8t+7 of two 32-row quarters) are to hit all 64 banks: rows of 256 bytes 16
// different slots (tr_swizzle); rows of 128 bytes, half the banks each, 8 different slots for the even rows and for the odd ones.
template <int WIDTH>
__device__ __forceinline__ int mid_tr_swizzle(int k) {
    if constexpr (WIDTH == 256) return tr_swizzle(k);
    else return ((k >> 1) & 3) | (((k >> 5) & 1) << 2);
}

// Byte offsets of the DMAs of a transposed operand of WIDTH rows: instruction d of wave w covers 1024 / WIDTH contraction rows.
template <int WIDTH>
__device__ __forceinline__ uint32_t mid_tr_voff(int instr, int64_t ld, int64_t unit, int first_block, int last_block) {
    constexpr int SLOTS = WIDTH / 16;
    const int lane = threadIdx.x & 63;
    const int row = instr * (64 / SLOTS) + lane / SLOTS;
    const int c = (lane % SLOTS) ^ mid_tr_swizzle<WIDTH>(row);
    const int blk = min(first_block + (c >> 2), last_block) - first_block;  // blocks past the edge re-read the last one
    return (uint32_t)(row * ld + blk * unit) + (c & 3) * 16;
}

// Workgroup `bid` of the `grid` that compute this product (or one part of its k).
// ODD_ROWS: rows of C start at odd multiples of two bytes too (see ShiftedRows); a piece is then stored behind the next one.
template <int AF, int BF, int C_DT, int TJ, bool A_TR, bool B_TR, bool ODD_ROWS, bool BIAS_AFTER = false>
__device__ __forceinline__ void gemm_mid_tile(
    const int bid, const int grid, const int split, const uint8_t* __restrict__ A, int64_t lda, int64_t a_unit, const uint8_t* __restrict__ Bt,
    int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa_dev, const float* sb_dev, void* __restrict__ C,
    int64_t ldc, const void* __restrict__ bias, int tiles_m, int tiles_n, int c_vec_ok, int k_splits, int bias_fp32 = 0) {
    using Cfg = MidCfg<TJ>;
    constexpr int NSTAGE = Cfg::NSTAGE, NDMA = Cfg::NDMA;
    extern __shared__ __align__(16) uint8_t smem[];
    // consecutive workgroup ids go to the 8 XCDs round-robin; re-deal them so that one XCD (one L2) gets a contiguous
    // run of the tile order, which walks bands of eight tile rows column by column: the 32 workgroups of an XCD then
    // hold a patch of 8 x 4 neighbouring tiles, the fewest operand panels through that L2
    const int lid = xcd_contiguous_id(bid, grid);
    const int band = lid / (8 * tiles_n), in_band = lid % (8 * tiles_n);
    const int band_rows = min(tiles_m - band * 8, 8);
    const int tm = band * 8 + in_band % band_rows, tn = in_band / band_rows;
    const int m0 = tm * MID_TILE_M, n0 = tn * Cfg::TILE_N;
    // k_splits > 1 (host: fp32 output, no bias): takes the split-th part of k and writes its partial sums,
    // unscaled, to the split-th M x ldc slab of C; a second kernel adds the slabs in a fixed order.
    const int K_part = K / k_splits;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 1, wn = wave & 1;

    // ---- DMA: one instruction = 16 rows x 64 B of one unit, landing as 1 KB of consecutive LDS; lane l fetches
    // row l/4 of the sixteen, piece (l%4) ^ (l/32) (the slot swizzle, applied on the global side).  Wave w
    // brings row groups 2w, 2w+1 of both units of A and BI*w .. BI*w+BI-1 of both units of Bt.
    const uint32_t lds_u32 = (uint32_t)(uintptr_t)smem;
    // Transposed operand: instruction d of a wave's 4 (128 rows) or 8 (256 rows) brings 8 or 4 whole contraction rows.
    constexpr int A_VOFF = A_TR ? 4 : 2, B_VOFF = B_TR ? 2 * Cfg::BI : Cfg::BI;
    uint32_t a_voff[A_VOFF], b_voff[B_VOFF];
    const uint32_t piece = (uint32_t)(((lane & 3) ^ (lane >> 5)) << 4);
#pragma unroll
    for (int i = 0; i < A_VOFF; i++) {
        if constexpr (A_TR) a_voff[i] = mid_tr_voff<MID_TILE_M>(wave * 4 + i, lda, a_unit, m0 / 64, M / 64 - 1);
        else a_voff[i] = (uint32_t)(min((wave * 2 + i) * 16 + (lane >> 2), M - 1 - m0) * lda) + piece;  // rows past the edge re-read the last row
    }
#pragma unroll
    for (int i = 0; i < B_VOFF; i++) {
        if constexpr (B_TR) b_voff[i] = mid_tr_voff<Cfg::TILE_N>(wave * 2 * Cfg::BI + i, ldb, b_unit, n0 / 64, N / 64 - 1);
        else b_voff[i] = (uint32_t)(min((wave * Cfg::BI + i) * 16 + (lane >> 2), N - 1 - n0) * ldb) + piece;
    }
    const int64_t k0 = (int64_t)split * K_part;
    const uint8_t* a_ptr = A_TR ? A + (int64_t)(m0 / 64) * a_unit + k0 * lda : A + (int64_t)m0 * lda + k0 / 64 * a_unit;
    const uint8_t* b_ptr = B_TR ? Bt + (int64_t)(n0 / 64) * b_unit + k0 * ldb : Bt + (int64_t)n0 * ldb + k0 / 64 * b_unit;
    // DMA d = 0..NDMA-1 of this wave's share of a step (4 of A, then Bt); the pointers move on after the last
    auto issue1 = [&](uint32_t base, int d) __attribute__((always_inline)) {
        if (d < 4) {
            if constexpr (A_TR) dma_mid(a_ptr, a_voff[d], base + (wave * 4 + d) * 1024);
            else dma_mid(a_ptr + (d >> 1) * a_unit, a_voff[d & 1], base + (d >> 1) * MID_A_UNIT + (wave * 2 + (d & 1)) * 1024);
        } else {
            const int h = (d - 4) / Cfg::BI, i = (d - 4) % Cfg::BI;
            if constexpr (B_TR) dma_mid(b_ptr, b_voff[d - 4], base + 2 * MID_A_UNIT + (wave * 2 * Cfg::BI + d - 4) * 1024);
            else dma_mid(b_ptr + h * b_unit, b_voff[i], base + 2 * MID_A_UNIT + h * Cfg::B_UNIT + (wave * Cfg::BI + i) * 1024);
        }
        if (d == NDMA - 1) {
            a_ptr += A_TR ? 128 * lda : 2 * a_unit;
            b_ptr += B_TR ? 128 * ldb : 2 * b_unit;
        }
    };

    // ---- fragments: lane -> tile row lane % 16, k quarter lane / 16 (32 bytes = two 16-byte pieces of one unit)
    const int frow = lane & 15, fq = lane >> 4;
    const int fsw = (frow >> 3) & 1;
    const int f_row0 = frow * 64 + ((((fq & 1) * 2 + 0) ^ fsw) << 4);
    const int f_row1 = frow * 64 + ((((fq & 1) * 2 + 1) ^ fsw) << 4);
    const int fa_off = (fq >> 1) * MID_A_UNIT + wm * 64 * 64;
    const int fb_off = 2 * MID_A_UNIT + (fq >> 1) * Cfg::B_UNIT + wn * (TJ * 16) * 64;

    v4f_m acc[TJ][4];  // [tj][ti]
#pragma unroll
    for (int tj = 0; tj < TJ; tj++)
#pragma unroll
        for (int ti = 0; ti < 4; ti++) acc[tj][ti] = (v4f_m){0.f, 0.f, 0.f, 0.f};
    v8i fa[2][4], fb[2][TJ];  // [parity of the step]: one step's fragments are multiplied while the next one's are read
    // transposed operand: lane j of a 16-lane group q addresses contraction row 32q + 8t + j/2 (t-th read), byte column
    // tile*16 + 8*(j%2), through the slot swizzle (the same for all four reads of a lane)
    const int tr_row = 32 * fq + (frow >> 1);
    const int a_tr0 = tr_row * MID_TILE_M + 8 * (frow & 1), a_trf = mid_tr_swizzle<MID_TILE_M>(tr_row);
    const int b_tr0 = 2 * MID_A_UNIT + tr_row * Cfg::TILE_N + 8 * (frow & 1), b_trf = mid_tr_swizzle<Cfg::TILE_N>(tr_row);
    auto frag_a = [&](const uint8_t* st, int t) __attribute__((always_inline)) {
        if constexpr (A_TR) {
            return read_frag_tr<MID_TILE_M>(st + a_tr0 + (((wm * 4 + t) ^ a_trf) << 4));
        } else {
            const uint8_t* p = st + fa_off + t * 16 * 64;
            return read_frag(p + f_row0, p + f_row1);
        }
    };
    auto frag_b = [&](const uint8_t* st, int t) __attribute__((always_inline)) {
        if constexpr (B_TR) {
            return read_frag_tr<Cfg::TILE_N>(st + b_tr0 + (((wn * TJ + t) ^ b_trf) << 4));
        } else {
            const uint8_t* p = st + fb_off + t * 16 * 64;
            return read_frag(p + f_row0, p + f_row1);
        }
    };
    // all fragments of the first step into set P
    auto fetch_all = [&](auto parity) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value;
#pragma unroll
        for (int t = 0; t < 4; t++) fa[P][t] = frag_a(smem, t);
#pragma unroll
        for (int t = 0; t < TJ; t++) fb[P][t] = frag_b(smem, t);
    };
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    constexpr std::integral_constant<int, 2> c2{};
    constexpr std::integral_constant<int, 3> c3{};

    const int steps = K_part / 128;
    // prologue: every stage is filled, step 0's fragments are read.  The parity of a step is that of its distance to
    // the last one, so that the tail of the loop below is the same code for every k.
#pragma unroll
    for (int p = 0; p < NSTAGE; p++)
        if (p < steps) {
#pragma unroll
            for (int d = 0; d < NDMA; d++) issue1(lds_u32 + p * Cfg::STAGE, d);
        }
    // 1 / (sa * sb) for the epilogue, kept in a scalar register.  The scales are asked for behind the DMAs (the pointers
    // pass through the asm, which keeps the compiler from moving the loads up): asked for first, the DMAs waited a
    // round trip to memory for them
    asm volatile("" : "+s"(sa_dev), "+s"(sb_dev)::"memory");
    const float inv = k_splits > 1 ? 1.0f : __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(
        int, __fdiv_rn(1.0f, load_scalar(sa_dev)) * __fdiv_rn(1.0f, load_scalar(sb_dev)))));
    // step 0's data is there; what was asked for behind it, min(steps, NSTAGE) - 1 steps, may still be in flight (with fewer steps than
    // stages too: waiting for all of it cost 512-deep products of many columns a tenth, 17 rows, 28672 x 512: 7.8 / 7.25 us)
    if (steps >= NSTAGE) mid_wait_barrier<(NSTAGE - 1) * NDMA>();
    else if (NSTAGE == 5 && steps == 4) mid_wait_barrier<3 * NDMA>();
    else if (NSTAGE == 5 && steps == 3) mid_wait_barrier<2 * NDMA>();
    else if (steps == 2) mid_wait_barrier<NDMA>();
    else mid_wait_barrier<0>();
    if (steps & 1) fetch_all(c0);
    else fetch_all(c1);

    // ---- epilogue: MFMA(first = Bt rows, second = A rows) leaves lane l with row ti*16 + l%16 and the four
    // columns tj*16 + 4*(l/16) + e of the wave's 64 x (16 TJ)
    const int lm = lane & 15, lq = lane >> 4;
    const int wcol0 = n0 + wn * (TJ * 16);
    float bv[TJ][4];
    // 2-byte outputs, one store instruction at a time: rows ti*16 .. +15, columns tp*32 .. +31 of the wave's part.
    // v_permlane16_swap between the accumulator tiles 2p and 2p + 1 trades the odd 16-lane rows of the first for the
    // even ones of the second, which turns a lane's 4 + 4 columns of two tiles into 8 neighbouring columns of one (lq
    // even: columns 4 lq .. + 7 of tile 2p, lq odd: 4 (lq - 1) .. + 7 of tile 2p + 1): one 16-byte store per lane, 64
    // contiguous bytes per row and instruction.
    ShiftedRows rows_shifted(C, ldc, m0 + wm * 64 + lm);
    const bool whole = m0 + MID_TILE_M <= M && n0 + Cfg::TILE_N <= N;
    const bool interior = c_vec_ok && whole;  // the same for every lane: nothing to check
    const int col_l = wcol0 + (lq & 1) * 16 + (lq >> 1) * 8;
    float* const base32 = (float*)C + ((int64_t)split * M + m0 + wm * 64 + lm) * ldc + wcol0 + 4 * lq;  // of the lane's first piece of an fp32 C
    auto store_held = [&](int ti, int tp) __attribute__((always_inline)) {
        const int row = m0 + wm * 64 + ti * 16 + lm, col = col_l + tp * 32;
        uint16_t* dst = (uint16_t*)C + (int64_t)row * ldc + col;
        if (whole) rows_shifted.store(dst, true, tp == 0, tp == TJ / 2 - 1, 0, 0, M, N);
        else rows_shifted.store(dst, false, tp == 0, tp == TJ / 2 - 1, row, col, M, N);
    };
    auto store_piece = [&](int ti, int tp) __attribute__((always_inline)) {
        const int te = 2 * tp, to = 2 * tp + 1;
        if constexpr (c_is_fp32(C_DT)) {  // a lane's 4 columns are 16 bytes already
            const int row = m0 + wm * 64 + ti * 16 + lm, col = wcol0 + te * 16 + 4 * lq;
            float* dst = base32 + ((int64_t)(ti * 16) * ldc + tp * 32);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const float v[4] = {acc[te + h][ti][0], acc[te + h][ti][1], acc[te + h][ti][2], acc[te + h][ti][3]};
                store_fp32x4(dst + 16 * h, finish4<C_DT, BIAS_AFTER>(v, inv, bv[te + h]), interior, c_vec_ok, row, col + 16 * h, M, N);
            }
        } else {
            const uint32_t x0 = finish2<C_DT, BIAS_AFTER>(acc[te][ti][0], acc[te][ti][1], inv, bv[te][0], bv[te][1]);
            const uint32_t x1 = finish2<C_DT, BIAS_AFTER>(acc[te][ti][2], acc[te][ti][3], inv, bv[te][2], bv[te][3]);
            const uint32_t y0 = finish2<C_DT, BIAS_AFTER>(acc[to][ti][0], acc[to][ti][1], inv, bv[to][0], bv[to][1]);
            const uint32_t y1 = finish2<C_DT, BIAS_AFTER>(acc[to][ti][2], acc[to][ti][3], inv, bv[to][2], bv[to][3]);
            const auto s0 = __builtin_amdgcn_permlane16_swap(x0, y0, false, false);  // every lane takes part
            const auto s1 = __builtin_amdgcn_permlane16_swap(x1, y1, false, false);
            if constexpr (ODD_ROWS) {
                if (tp > 0) store_held(ti, tp - 1);
                else if (ti > 0) store_held(ti - 1, TJ / 2 - 1);
                rows_shifted.hold(make_uint4(s0[0], s1[0], s0[1], s1[1]));
                return;
            }
            const int row = m0 + wm * 64 + ti * 16 + lm, col = col_l + tp * 32;
            uint16_t* dst = (uint16_t*)C + (int64_t)row * ldc + col;
            if (__builtin_expect(interior, 1)) {
                store16_any(dst, make_uint4(s0[0], s1[0], s0[1], s1[1]));
            } else if (row < M && col < N) {
                if (c_vec_ok && col + 8 <= N) {
                    store16_any(dst, make_uint4(s0[0], s1[0], s0[1], s1[1]));
                } else {
                    const uint32_t w[4] = {s0[0], s1[0], s0[1], s1[1]};
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (col + e < N) dst[e] = (uint16_t)((w[e >> 1] >> (16 * (e & 1))) & 0xffffu);
                }
            }
        }
    };
    int cur = 0;  // stage of step s
    // One step: its products, between them the reads of the next step's fragments and the DMAs of the step NSTAGE
    // ahead into the stage whose fragments every wave holds by now.  IN_FLIGHT: steps that may still be in flight once
    // the next step's data is there.  MODE 0: both exist; 1: nothing left to fetch; 2: last step.
    auto step = [&](auto parity, auto mode, auto in_flight) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value, MODE = decltype(mode)::value;
        const int next = cur + 1 == NSTAGE ? 0 : cur + 1;
        const uint8_t* st = smem + next * Cfg::STAGE;
        const uint32_t refill = lds_u32 + cur * Cfg::STAGE;
        // everybody's DMAs of step s+1 have landed and everybody's reads of this step's stage are done
        if constexpr (MODE < 2) mid_wait_barrier<decltype(in_flight)::value * NDMA>();
        if constexpr (MODE == 2) {
            if constexpr (c_is_fp32(C_DT)) load_bias_tiles<F8MI_FP32, TJ>(bv, bias, wcol0 + 4 * lq, N);
            else if constexpr (BIAS_AFTER) load_rounded_bias_tiles<C_DT, TJ>(bv, bias, bias_fp32, wcol0 + 4 * lq, N);
            else load_bias_tiles<C_DT, TJ>(bv, bias, wcol0 + 4 * lq, N);
        }
        F8MI_SCHED_FENCE();
#pragma unroll
        for (int ti = 0; ti < 4; ti++)
#pragma unroll
            for (int tj = 0; tj < TJ; tj++) {
                const int i = ti * TJ + tj;
                acc[tj][ti] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[P][tj], fa[P][ti], acc[tj][ti], BF, AF, 0, 0, 0, 0);
                if constexpr (MODE < 2) {
                    F8MI_SCHED_FENCE();
                    if (MODE == 0 && (i & 1) && i / 2 < NDMA) issue1(refill, i / 2);
                    if ((i & 1) == 0) {
                        const int f = i / 2;
                        if (f == 0) fa[P ^ 1][0] = frag_a(st, 0);
                        else if (f <= TJ) fb[P ^ 1][f - 1] = frag_b(st, f - 1);
                        else if (f < TJ + 4) fa[P ^ 1][f - TJ] = frag_a(st, f - TJ);
                    }
                    F8MI_SCHED_FENCE();
                } else if (ti >= 1 && (tj & 1)) {  // the finished row of tiles, under this row's products
                    F8MI_SCHED_FENCE();
                    store_piece(ti - 1, tj >> 1);
                    F8MI_SCHED_FENCE();
                }
            }
        cur = next;
    };
    constexpr std::integral_constant<int, NSTAGE - 2> steady{};
    int n_steady = steps - NSTAGE;  // steps that fetch
    if (n_steady > 0 && (n_steady & 1)) { step(c1, c0, steady); n_steady--; }
    for (; n_steady > 0; n_steady -= 2) {
        step(c0, c0, steady);
        step(c1, c0, steady);
    }
    if constexpr (NSTAGE == 5) {
        if (steps >= 5) step(c0, c1, c3);
        if (steps >= 4) step(c1, c1, c2);
    }
    if (steps >= 3) step(c0, c1, c1);
    if (steps >= 2) step(c1, c1, c0);
    step(c0, c2, c0);

#pragma unroll
    for (int tp = 0; tp < TJ / 2; tp++) store_piece(3, tp);
    if constexpr (ODD_ROWS) store_held(3, TJ / 2 - 1);
}

template <int AF, int BF, int C_DT, int TJ, bool A_TR, bool B_TR, bool ODD_ROWS>
__global__ __launch_bounds__(GEMM_THREADS) void gemm_mid_kernel(
    const uint8_t* __restrict__ A, int64_t lda, int64_t a_unit, const uint8_t* __restrict__ Bt, int64_t ldb, int64_t b_unit,
    int M, int N, int K, const float* sa_dev, const float* sb_dev, void* __restrict__ C,
    int64_t ldc, const void* __restrict__ bias, int tiles_m, int tiles_n, int c_vec_ok, int k_splits) {
    gemm_mid_tile<AF, BF, C_DT, TJ, A_TR, B_TR, ODD_ROWS>(blockIdx.x, gridDim.x, blockIdx.y, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa_dev, sb_dev, C,
                                                          ldc, bias, tiles_m, tiles_n, c_vec_ok, k_splits);
}

template <int AF, int BF, int C_DT, int TJ, bool A_TR, bool B_TR, bool ODD_ROWS>
static int launch_mid4(hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit, const uint8_t* Bt, int64_t ldb,
                       int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C, int64_t ldc, const void* bias,
                       int c_vec_ok, int k_splits) {
    static std::atomic<uint64_t> lds_allowed{0};
    auto kern = gemm_mid_kernel<AF, BF, C_DT, TJ, A_TR, B_TR, ODD_ROWS>;
    if (int rc = allow_big_lds(kern, MidCfg<TJ>::LDS, lds_allowed)) return rc;
    const int tiles_m = (M + MID_TILE_M - 1) / MID_TILE_M, tiles_n = (N + MidCfg<TJ>::TILE_N - 1) / MidCfg<TJ>::TILE_N;
    hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n), (unsigned)k_splits), dim3(GEMM_THREADS), MidCfg<TJ>::LDS, stream, A, lda, a_unit,
                       Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, tiles_m, tiles_n, c_vec_ok, k_splits);
    return check_hip(hipGetLastError(), "gemm (128-row tiles) kernel launch");
}

template <int AF, int BF, int C_DT, bool A_TR, bool B_TR, bool ODD_ROWS>
static int launch_mid3(bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit, const uint8_t* Bt, int64_t ldb,
                       int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C, int64_t ldc, const void* bias,
                       int c_vec_ok, int k_splits) {
    if (wide) return launch_mid4<AF, BF, C_DT, 8, A_TR, B_TR, ODD_ROWS>(stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
    return launch_mid4<AF, BF, C_DT, 4, A_TR, B_TR, ODD_ROWS>(stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
}

template <int AF, int BF, bool A_TR, bool B_TR, bool ODD_ROWS>
static int launch_mid2(int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit, const uint8_t* Bt,
                       int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C, int64_t ldc,
                       const void* bias, int c_vec_ok, int k_splits) {
    if (c_dtype == F8MI_BF16) return launch_mid3<AF, BF, F8MI_BF16, A_TR, B_TR, ODD_ROWS>(wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
    if (c_dtype == F8MI_FP16) return launch_mid3<AF, BF, F8MI_FP16, A_TR, B_TR, ODD_ROWS>(wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
    if constexpr (ODD_ROWS) { set_error("gemm: fp32 rows are never at odd multiples of two bytes"); return F8MI_ERR_INVALID_ARG; }
    else return launch_mid3<AF, BF, F8MI_FP32, A_TR, B_TR, false>(wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
}

template <bool A_TR, bool B_TR, bool ODD_ROWS = false>
static int launch_mid1(int a_fmt, int b_fmt, int c_dtype, bool wide, hipStream_t stream, const uint8_t* A, int64_t lda, int64_t a_unit,
                       const uint8_t* Bt, int64_t ldb, int64_t b_unit, int M, int N, int K, const float* sa, const float* sb, void* C,
                       int64_t ldc, const void* bias, int c_vec_ok, int k_splits) {
    if (a_fmt == F8MI_E4M3FN && b_fmt == F8MI_E4M3FN) return launch_mid2<0, 0, A_TR, B_TR, ODD_ROWS>(c_dtype, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
    if (a_fmt == F8MI_E5M2 && b_fmt == F8MI_E4M3FN) return launch_mid2<1, 0, A_TR, B_TR, ODD_ROWS>(c_dtype, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
    if (a_fmt == F8MI_E4M3FN && b_fmt == F8MI_E5M2) return launch_mid2<0, 1, A_TR, B_TR, ODD_ROWS>(c_dtype, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
    return launch_mid2<1, 1, A_TR, B_TR, ODD_ROWS>(c_dtype, wide, stream, A, lda, a_unit, Bt, ldb, b_unit, M, N, K, sa, sb, C, ldc, bias, c_vec_ok, k_splits);
}

}  // namespace f8mi
