// K2 / K2d: saturated fp8 cast, with the transposed copy and (optionally) the
// tensor's amax fused into the same pass.  HBM-bound: reads sizeof(T) bytes and
// writes 1 byte per element and per fp8 output.
//
// A workgroup of 256 lanes owns a 128 x 128 tile.  Lane t covers columns
// 8*(t%16) .. +7 of rows 64*h + 4*(t/16) .. +3 for h = 0, 1: eight 16-byte loads
// (bf16/fp16; sixteen for fp32), all issued before the first use.  The row-major
// fp8 tile goes out straight from registers as 8-byte stores (16 lanes = one
// 128-byte row segment).  For the transposed copy each lane transposes its
// 4 x 8 byte block in registers (v_perm), parks the 4-row dwords in a
// 128 x 128-byte LDS tile whose dword index is XOR-swizzled by the column group
// (so the 64 lanes of a store hit 32 banks twice: the floor for 256 bytes), and
// the tile is read back as 16-byte row pieces: 8 lanes = one 128-byte segment of
// a row of the transposed output.
#include <algorithm>
#include <atomic>
#include <mutex>

#include "f8mi_cast_util.h"

namespace f8mi {

// The fp8 bytes leave as 8-byte (row-major copy) and 16-byte (transposed copy) stores at whatever alignment the
// output's row pitch gives them.
__device__ __forceinline__ void store8(uint8_t* p, uint32_t lo, uint32_t hi) {
#if F8MI_CAST_NT_STORES
    __builtin_nontemporal_store((u32x2){lo, hi}, (u32x2_any*)p);
#else
    store8_any(p, lo, hi);
#endif
}
__device__ __forceinline__ void store16(uint8_t* p, uint4 v) {
#if F8MI_CAST_NT_STORES
    __builtin_nontemporal_store((u32x4){v.x, v.y, v.z, v.w}, (u32x4_any*)p);
#else
    store16_any(p, v);
#endif
}

constexpr int CAST_THREADS = 256;
constexpr int SPREAD_WORDS = 1024;  // words of the delayed-scaling workspace (f8mi_delayed_workspace_bytes)
constexpr int CAST_TILE = 128;
constexpr int CAST_GROUP = 8;

// Fused amax of the cast kernel, without a workspace: *amax_out was zeroed by a tiny kernel launched just before, and holds the
// running maximum as an fp32 bit pattern (non-negative floats and NaNs order like unsigned integers).
// No ticket and, for all but a handful of blocks, no atomic at all: the value only grows, so a block whose
// maximum is not above a (possibly stale) read of it has nothing to add.  (Reducing and reading the word early, right
// after the loads, so that the round trip overlaps the conversion, was 20 % slower: the barrier it needs in the
// middle of the block makes all four waves wait for the slowest one's loads before any of them converts.)
__device__ __forceinline__ void publish_amax_cast(uint32_t blockmax, float* amax_out, int in_dt) {
    if (threadIdx.x == 0) {
        const uint32_t bits = __float_as_uint(abs_bits_to_float(blockmax, in_dt));
        uint32_t* dst = (uint32_t*)amax_out;
        if (bits > __atomic_load_n(dst, __ATOMIC_RELAXED)) atomicMax(dst, bits);
    }
}

// 4 dwords (rows 0..3, 4 bytes each = columns 0..3) -> 4 dwords (column c: rows 0..3)
__device__ __forceinline__ void transpose4x4_bytes(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3, uint32_t& c0,
                                                   uint32_t& c1, uint32_t& c2, uint32_t& c3) {
    // v_perm_b32(hi, lo, sel): byte i of the result = byte sel[i] of the 8-byte {hi,lo} (lo = bytes 0..3)
    uint32_t a = __builtin_amdgcn_perm(r1, r0, 0x05010400u);  // r0.b0 r1.b0 r0.b1 r1.b1
    uint32_t b = __builtin_amdgcn_perm(r1, r0, 0x07030602u);  // r0.b2 r1.b2 r0.b3 r1.b3
    uint32_t c = __builtin_amdgcn_perm(r3, r2, 0x05010400u);  // r2.b0 r3.b0 r2.b1 r3.b1
    uint32_t d = __builtin_amdgcn_perm(r3, r2, 0x07030602u);  // r2.b2 r3.b2 r2.b3 r3.b3
    c0 = __builtin_amdgcn_perm(c, a, 0x05040100u);            // a.b0 a.b1 c.b0 c.b1
    c1 = __builtin_amdgcn_perm(c, a, 0x07060302u);            // a.b2 a.b3 c.b2 c.b3
    c2 = __builtin_amdgcn_perm(d, b, 0x05040100u);
    c3 = __builtin_amdgcn_perm(d, b, 0x07060302u);
}

template <int DT>
struct Row8 {  // eight consecutive elements of one row, widened to fp32 on demand
    uint32_t w[DT == F8MI_FP32 ? 8 : 4];
};

template <int DT>
__device__ __forceinline__ float elem(const Row8<DT>& r, int i) {
    if constexpr (DT == F8MI_FP32) return __uint_as_float(r.w[i]);
    else {
        uint32_t h = (i & 1) ? (r.w[i >> 1] >> 16) : (r.w[i >> 1] & 0xffffu);
        if constexpr (DT == F8MI_BF16) return bf16_bits_to_float(h);
        else return fp16_bits_to_float(h);
    }
}

// Nothing of the row that is worked out before this is kept for what comes after it: on one side of a branch it keeps the compiler from
// unpacking the rows, which both sides do, ahead of it (16-bit cast with its maximum collected: 73 registers and six workgroups a CU, with
// this 61 and eight; 8192 x 4096 with both copies 31.2 -> 30.1 us).  Not fp32, where nothing is unpacked: five workgroups instead of four were slower.
template <int DT>
__device__ __forceinline__ void set_apart(Row8<DT>& r) {
#pragma unroll
    for (uint32_t& w : r.w) asm("" : "+v"(w));
}

// Folds the eight elements of a row into a running maximum.  16-bit types: `m` holds two 16-bit maxima side by side
// (see absmax16x2); absmax_done merges them.
template <int DT>
__device__ __forceinline__ uint32_t absmax_row(const Row8<DT>& r, uint32_t m) {
    if constexpr (DT == F8MI_FP32) {
#pragma unroll
        for (int i = 0; i < 8; i++) { uint32_t a = r.w[i] & 0x7fffffffu; m = m > a ? m : a; }
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++) m = absmax16x2(r.w[i], m);
    }
    return m;
}
template <int DT>
__device__ __forceinline__ uint32_t absmax_done(uint32_t m) {
    if constexpr (DT == F8MI_FP32) return m;
    else return fold16(m);
}

// Eight elements -> eight fp8 bytes.
template <int DT, int PROD, int FMT, bool WITHIN>
__device__ __forceinline__ void cast_row8(const Row8<DT>& r, float scale, uint32_t& lo, uint32_t& hi) {
    lo = cast4<PROD, FMT, WITHIN>(elem<DT>(r, 0), elem<DT>(r, 1), elem<DT>(r, 2), elem<DT>(r, 3), scale);
    hi = cast4<PROD, FMT, WITHIN>(elem<DT>(r, 4), elem<DT>(r, 5), elem<DT>(r, 6), elem<DT>(r, 7), scale);
}

// Loads 8 elements of row `row` starting at column `col`; out-of-range elements read as +0.  Eight elements inside the
// row are one 16-byte load (two for fp32) whatever the row pitch: a row only has to start at a multiple of the
// element size.
template <int DT>
__device__ __forceinline__ void load_row8(Row8<DT>& r, const void* x, int64_t row, int64_t col, int64_t rows,
                                          int64_t cols, int64_t ld) {
    constexpr int ESZ = DT == F8MI_FP32 ? 4 : 2;
    constexpr int NW = DT == F8MI_FP32 ? 8 : 4;
#pragma unroll
    for (int i = 0; i < NW; i++) r.w[i] = 0u;
    if (row >= rows || col >= cols) return;
    const char* p = (const char*)x + (row * ld + col) * ESZ;
    if (col + 8 <= cols) {
        uint4 v0 = load_nt16_any(p);
        r.w[0] = v0.x; r.w[1] = v0.y; r.w[2] = v0.z; r.w[3] = v0.w;
        if constexpr (DT == F8MI_FP32) {
            uint4 v1 = load_nt16_any(p + 16);
            r.w[4] = v1.x; r.w[5] = v1.y; r.w[6] = v1.z; r.w[7] = v1.w;
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; i++) {
            if (col + i < cols) {
                if constexpr (DT == F8MI_FP32) r.w[i] = ((const uint32_t*)p)[i];
                else r.w[i >> 1] |= (uint32_t)((const uint16_t*)p)[i] << ((i & 1) * 16);
            }
        }
    }
}

// Which tile (ty, tx) of a tiles_y x tiles_x grid workgroup `bid` of `nb` takes.  Tiles are walked in bands of CAST_GROUP tile
// rows and, inside a band, in groups of CAST_GROUP tile columns: the blocks in flight then read 2 KB runs of each input row
// and write 1 KB runs of each transposed row, instead of one of the two walking through memory with a huge stride.
__device__ __forceinline__ void cast_tile_of(uint32_t bid, uint32_t nb, uint32_t tiles_x, uint32_t tiles_y, int& ty, int& tx) {
    // Consecutive workgroup ids go to the 8 XCDs round-robin; re-deal them so that one XCD (one L2) gets whole
    // groups of 64 neighbouring tiles (an 8 x 8 supertile where the tile grid divides evenly) and can merge
    // their adjacent output segments, while consecutive groups go to consecutive XCDs: the workgroups in flight
    // on the whole chip then cover ONE contiguous stretch of the tensor that advances through memory.  (Giving
    // each XCD its own eighth of the tensor instead, eight fronts far apart, measured 5 % slower in the
    // benchmark step: 5.36 -> 5.63 TB/s; up to 20 % on tensors below 300 MB.)
    // (32-bit arithmetic: the host has checked that the tiles number at most 2^31 - 1; the 64-bit divisions of before cost every
    // workgroup 0.4 us: 8192 x 4096 with both copies 30.6 -> 28.2 us, 16 x 4096 4.7 -> 4.3)
    const uint32_t nb_full = nb - nb % 512;  // ids past the last whole round of 8 groups stay
    if (bid < nb_full) {
        const uint32_t xcd = bid % 8, j = bid / 8;
        bid = ((j / 64) * 8 + xcd) * 64 + (j % 64);
    }
#if F8MI_CAST_REVERSE_WALK  // measurement builds only: last tiles first, the reverse of the order the amax pass read in
    bid = nb - 1 - bid;
#endif
    const uint32_t band = tiles_y <= CAST_GROUP ? 0 : bid / (CAST_GROUP * tiles_x);  // (one band: the product may not fit)
    const uint32_t rem = bid - band * CAST_GROUP * tiles_x;
    const uint32_t rows_in_band = min((uint32_t)CAST_GROUP, tiles_y - band * CAST_GROUP);
    const uint32_t gcol = rem / (rows_in_band * CAST_GROUP);
    const uint32_t r2 = rem - gcol * rows_in_band * CAST_GROUP;
    const uint32_t cols_in_g = min((uint32_t)CAST_GROUP, tiles_x - gcol * CAST_GROUP);
    ty = (int)(band * CAST_GROUP + r2 / cols_in_g);
    tx = (int)(gcol * CAST_GROUP + r2 % cols_in_g);
}

// A tile of 64 H rows x 128 columns at (r0, c0), one per workgroup of 256 lanes: lane t holds columns 8 (t % 16) .. + 7 of rows
// 64 h + 4 (t / 16) .. + 3 for h < H.
template <int DT, int H>
__device__ __forceinline__ void load_tile(Row8<DT> (&in)[H][4], const void* x, int64_t r0, int64_t c0, int64_t rows, int64_t cols, int64_t ld) {
    const int a = threadIdx.x & 15, b = threadIdx.x >> 4;
#pragma unroll
    for (int h = 0; h < H; h++)
#pragma unroll
        for (int j = 0; j < 4; j++) load_row8<DT>(in[h][j], x, r0 + 64 * h + 4 * b + j, c0 + 8 * a, rows, cols, ld);
}
template <int DT, int H>
__device__ __forceinline__ uint32_t absmax_tile(const Row8<DT> (&in)[H][4]) {
    uint32_t m = 0;
#pragma unroll
    for (int h = 0; h < H; h++)
#pragma unroll
        for (int j = 0; j < 4; j++) m = absmax_row<DT>(in[h][j], m);
    return absmax_done<DT>(m);
}

// Scales, converts and stores such a tile: `out` row by row from registers, `out_t` through tileT.  out_kb / out_t_kb:
// F8MI_LAYOUT_* code of the respective output.  within (the same for the whole wave): within_range holds for all of it.
template <int DT, int PROD, int FMT, int H>
__device__ __forceinline__ void emit_tile(const Row8<DT> (&in)[H][4], uint32_t* tileT, float scale, bool within, int64_t r0, int64_t c0, int64_t rows, int64_t cols,
                                          uint8_t* __restrict__ out, uint8_t* __restrict__ out_t, int out_kb, int out_t_kb) {
    constexpr int DWORDS = 16 * H;                  // of a tile column: four rows each
    constexpr int SWIZZLE = 4 * H - 1;              // 16-byte pieces of a tile column, less one
    const int t = threadIdx.x;
    const int a = t & 15, b = t >> 4;
    const int64_t col = c0 + 8 * a;
    // Zero-padded k-blocked outputs (F8MI_LAYOUT_KBLOCK64_PAD128): the tile grid ends exactly where the padding does, so
    // a tile writes all of its columns (`out`) or rows (`out_t`); what lies past the tensor's edge is forced to
    // zero bytes (elements read as +0 would become NaN codes under a NaN scale).
    const bool pad = out_kb == F8MI_LAYOUT_KBLOCK64_PAD128 || out_t_kb == F8MI_LAYOUT_KBLOCK64_PAD128;
    uint32_t keep_lo = 0xffffffffu, keep_hi = 0xffffffffu;  // bytes of the lane's eight columns that lie inside the row
    if (pad && col + 8 > cols) {
        const int valid = col < cols ? (int)(cols - col) : 0;
        keep_lo = valid >= 4 ? 0xffffffffu : (valid ? (1u << (8 * valid)) - 1u : 0u);
        keep_hi = valid > 4 ? (1u << (8 * (valid - 4))) - 1u : 0u;
    }
#pragma unroll
    for (int h = 0; h < H; h++) {
        uint32_t lo[4], hi[4];
        if (within) {
#pragma unroll
            for (int j = 0; j < 4; j++) cast_row8<DT, PROD, FMT, true>(in[h][j], scale, lo[j], hi[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                Row8<DT> r = in[h][j];
                if constexpr (DT != F8MI_FP32) set_apart(r);
                cast_row8<DT, PROD, FMT, false>(r, scale, lo[j], hi[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int64_t row = r0 + 64 * h + 4 * b + j;
            if (pad) {
                lo[j] = row < rows ? lo[j] & keep_lo : 0u;
                hi[j] = row < rows ? hi[j] & keep_hi : 0u;
            }
            if (out && row < rows && (col < cols || out_kb == F8MI_LAYOUT_KBLOCK64_PAD128)) {
                // k-blocked: [cols/64][rows][64] (cols % 64 == 0 or padded to it: the eight columns are always whole)
                uint8_t* p = out_kb ? out + ((col >> 6) * rows + row) * 64 + (col & 63) : out + row * cols + col;
                if (out_kb || col + 8 <= cols) {
                    store8(p, lo[j], hi[j]);
                } else {
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (col + i < cols) p[i] = (uint8_t)((i < 4 ? lo[j] >> (8 * i) : hi[j] >> (8 * (i - 4))) & 0xffu);
                }
            }
        }
        if (out_t) {
            uint32_t tc[8];
            transpose4x4_bytes(lo[0], lo[1], lo[2], lo[3], tc[0], tc[1], tc[2], tc[3]);
            transpose4x4_bytes(hi[0], hi[1], hi[2], hi[3], tc[4], tc[5], tc[6], tc[7]);
            const int d = 16 * h + b;                    // dword index (rows 4d .. 4d+3) within a tile column
            const int dsw = d ^ ((a & SWIZZLE) << 2);    // swizzle by column group
#pragma unroll
            for (int cc = 0; cc < 8; cc++) tileT[(8 * a + cc) * DWORDS + dsw] = tc[cc];
        }
    }

    if (out_t) {
        __syncthreads();
#pragma unroll
        for (int p = 0; p < 2 * H; p++) {
            const int id = p * CAST_THREADS + t;
            const int c = id / (4 * H), q = id % (4 * H);  // tile column c (a row of out_t), 16-byte piece q
            const int qsw = q ^ ((c >> 3) & SWIZZLE);
            const uint4 v = *(const uint4*)&tileT[c * DWORDS + 4 * qsw];
            const int64_t gc = c0 + c;
            const int64_t gr = r0 + 16 * q;
            if (gc < cols && (gr < rows || out_t_kb == F8MI_LAYOUT_KBLOCK64_PAD128)) {
                // k-blocked: [rows/64][cols][64] (rows % 64 == 0 or padded to it: the sixteen rows are always whole)
                uint8_t* dst = out_t_kb ? out_t + ((gr >> 6) * cols + gc) * 64 + (gr & 63) : out_t + gc * rows + gr;
                if (out_t_kb || gr + 16 <= rows) {
                    store16(dst, v);
                } else {
                    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        if (gr + i < rows) dst[i] = (uint8_t)((w[i >> 2] >> (8 * (i & 3))) & 0xffu);
                }
            }
        }
    }
}

// An exchange of maxima inside a launch.  Whoever has one publishes a 64-bit word, {launch tag, maximum}, with an agent-scope store;
// whoever needs them all reads the words with agent-scope loads until each carries the tag: the words are all there is to
// exchange, so no fence is needed.  The tag is the host's count of such launches, so a word of any other launch
// just reads as "not there yet" and nothing has to be cleared; the host keeps launches that may run at the same time (other
// streams) on other words.  (The count has 32 bits: a word would be taken for a later launch's if exactly 2^32 launches had gone by
// without one that wrote it.)  Nothing depends on the others being on the chip: a workgroup that has waited for wait_ticks of the 100
// MHz clock reads the tiles whose words are missing itself.  So every wave ends whatever else runs, and the result is the same
// bits either way.
struct TaggedWords {
    uint64_t* words;  // null: no exchange
    uint32_t tag, wait_ticks;
};
// Everybody collects, and waits for workgroups that may find no room.  60 us: the last tile of the largest tensor arrives after 10 - 20, with
// as large a cast beside it after 40.  us a cast of 4096 x 4096 where two / three of them run at once on streams of their own, bf16: waits of
// 20: 17 / 38, 50 - 500: 16 / 21 (in turn on one stream: 18); fp32: 20: 50 / 61, 50: 25 / 65, 120: 24 / 83, 500: 24 / 242 (in turn: 25).
constexpr uint32_t EXCHANGE_WAIT_TICKS = 6000;
// Only the workgroup started last collects: the others end whatever it does, and most of them have.
constexpr uint32_t EXCHANGE_WAIT_TICKS_LAST = 200000;

__device__ __forceinline__ void publish_word(const TaggedWords& e, uint32_t i, uint32_t m) {
    __hip_atomic_store(&e.words[i], (uint64_t)e.tag << 32 | m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One tensor of a launch, as the kernels take it.
struct CastJob {
    const void* x;
    int64_t rows, cols, ld;
    uint8_t *out, *out_t;
    uint32_t tiles_x, tiles_y;
    int out_kb, out_t_kb;      // F8MI_LAYOUT_* code of the respective output
    const float* scale_dev;    // the scale, given beforehand; else
    float* scale_out;          // where the one found here goes,
    const uint32_t* amax_ws;   // found from the amax_nblocks maxima in amax_ws (the resident kernel: from the tensor itself)
    int amax_nblocks;
    float* amax_out;           // fused amax: its value, through
    uint32_t* amax_spread;     // these words, or
    TaggedWords tagged;        // an exchange
};

// The maximum of the tensor's n tiles of 64 H rows for a workgroup that has waited long enough: words that are there are taken, the
// tiles of those that are not are read, one after the other, each followed by another look at the words.  Workgroups start at
// different words and pick different tiles, and what one finds it publishes, so that together they read each missing tile about once
// (4096 x 4096, nobody waits at all: bf16 25 us for 16, fp32 53 for 24; when each of them read the whole tensor: 13.8 ms, bf16).  Every turn settles a word
// that was not: at most one for each word, whatever happens to the words meanwhile.  red: five words.
template <int DT, int H>
__device__ __forceinline__ uint32_t collect_late(const CastJob& j, uint32_t bid, uint32_t n, uint32_t* red) {
    const uint32_t t = threadIdx.x, wave = t >> 6;
    constexpr int ROWS = 4;  // loads at a time
    const uint32_t first = (bid * 0x9e3779b1u) % n;
    uint32_t m = 0;
    for (uint32_t k = 0; k < n; k += CAST_THREADS) {
        const bool mine = k + t < n;
        const uint32_t i = first + k + t < n ? first + k + t : first + k + t - n;
        bool settled = !mine;
        for (uint32_t turn = bid;; turn++) {
            if (!settled) {
                const uint64_t w = __hip_atomic_load(&j.tagged.words[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if ((uint32_t)(w >> 32) == j.tagged.tag) {
                    m = max(m, (uint32_t)w);
                    settled = true;
                }
            }
            const uint64_t missing = __ballot(!settled);
            __syncthreads();  // everybody has read `red`
            if ((t & 63) == 0) red[wave] = (uint32_t)__popcll(missing);
            __syncthreads();
            const uint32_t total = red[0] + red[1] + red[2] + red[3];
            if (!total) break;
            uint32_t rank = (uint32_t)__popcll(missing & ((1ull << (t & 63)) - 1));
            for (uint32_t v = 0; v < wave; v++) rank += red[v];
            if (!settled && rank == (turn * 0x85ebca6bu >> 8) % total) red[4] = i;
            __syncthreads();
            const uint32_t tile = red[4];
            if (mine && i == tile) settled = true;
            int ty, tx;
            cast_tile_of(tile, n, j.tiles_x, j.tiles_y, ty, tx);
            uint32_t found = 0;
#pragma unroll 1
            for (int r0 = t >> 4; r0 < 64 * H; r0 += 16 * ROWS) {
                Row8<DT> in[ROWS];
#pragma unroll
                for (int r = 0; r < ROWS; r++)
                    load_row8<DT>(in[r], j.x, (int64_t)ty * (64 * H) + r0 + 16 * r, (int64_t)tx * CAST_TILE + 8 * (t & 15), j.rows, j.cols, j.ld);
#pragma unroll
                for (int r = 0; r < ROWS; r++) found = absmax_row<DT>(in[r], found);
            }
            found = wave_max_u32(absmax_done<DT>(found));
            m = max(m, found);
            __syncthreads();  // everybody has read `red`
            if ((t & 63) == 0) red[wave] = found;
            __syncthreads();
            if (t == 0) publish_word(j.tagged, tile, max(max(red[0], red[1]), max(red[2], red[3])));
        }
    }
    m = wave_max_u32(m);
    __syncthreads();
    if ((t & 63) == 0) red[wave] = m;
    __syncthreads();
    return max(max(red[0], red[1]), max(red[2], red[3]));
}

// The same where only this workgroup collects, and the others, who wait for nobody, have left their words unless they were held up for
// as long as that: the whole tensor, in little code.
template <int DT>
__device__ __forceinline__ uint32_t collect_alone(const CastJob& j, uint32_t* red) {
    const int t = threadIdx.x;
    uint32_t m = 0;
    for (int64_t r = 0; r < (j.ld ? j.rows : 1); r++)
        for (int64_t c = 8 * t; c < j.cols; c += 8 * CAST_THREADS) {
            Row8<DT> v;
            load_row8<DT>(v, j.x, r, c, j.rows, j.cols, j.ld);
            m = absmax_row<DT>(v, m);
        }
    m = wave_max_u32(absmax_done<DT>(m));
    __syncthreads();  // everybody has read `red`
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    return max(max(red[0], red[1]), max(red[2], red[3]));
}

// Whether all n words were there in time; m: their maximum and every lane's, the same in all lanes of the workgroup.
// Every lane asks for BATCH words at a time, from the last ones (which come last) down: one round trip to memory (0.7 us) for each
// batch.  With every workgroup collecting, BATCH is 1: more words polled at a time hold up the loads that are waited for (4096 x 4096
// bf16: 18.9 us, with four 24.7).
template <int BATCH>
__device__ __forceinline__ bool collect_words(const TaggedWords& e, uint32_t n, uint32_t& m, uint32_t* red) {
    const int t = threadIdx.x;
    const uint64_t start = wall_clock64();
    constexpr uint32_t STEP = BATCH * CAST_THREADS, LATE = 0x80000000u;  // no maximum has the top bit
    for (uint32_t left = (n + STEP - 1) / STEP; left > 0 && !(m & LATE); left--) {
        const uint32_t i = (left - 1) * STEP + t;
        uint64_t w[BATCH];
        for (;;) {
            bool all = true;
#pragma unroll
            for (int u = 0; u < BATCH; u++)  // past the end: the last word again
                w[u] = __hip_atomic_load(&e.words[min(i + u * CAST_THREADS, n - 1)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int u = 0; u < BATCH; u++) all &= (uint32_t)(w[u] >> 32) == e.tag;
            if (all) break;
            if (wall_clock64() - start >= e.wait_ticks) { m |= LATE; break; }
            __builtin_amdgcn_s_sleep(1);
        }
#pragma unroll
        for (int u = 0; u < BATCH; u++) m = max(m, (uint32_t)w[u]);
    }
    static_assert(CAST_THREADS == 256, "four waves");
    m = wave_max_u32(m);
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    m = max(max(red[0], red[1]), max(red[2], red[3]));
    return !(m & LATE);
}

// Workgroup `bid` of the `nb` that cast the tensor.
template <int DT, int PROD, int FMT, bool TAGGED>
__device__ __forceinline__ void cast_body(const CastJob& j, uint32_t bid, uint32_t nb, uint32_t* tileT, uint32_t* red) {
    const void* const x = j.x;
    const int64_t rows = j.rows, cols = j.cols, ld = j.ld;
    float* const amax_out = j.amax_out;
    const uint32_t* const amax_ws = j.amax_ws;
    const int amax_nblocks = j.amax_nblocks;
    const int t = threadIdx.x;
    int ty, tx;
    cast_tile_of(bid, nb, j.tiles_x, j.tiles_y, ty, tx);
    const int64_t r0 = (int64_t)ty * CAST_TILE;
    const int64_t c0 = (int64_t)tx * CAST_TILE;

    // dynamic scaling: the amax kernel's per-workgroup maxima (at most WS_WORDS = 4 x 64 lanes x 4 words), requested
    // ahead of the tile so that they arrive first.  Every wave fetches all of them: no LDS, no barrier.
    static_assert(WS_WORDS <= 4 * 64 * 4, "four 16-byte loads per lane cover the workspace");
    uint4 ws_words[4];
    if (amax_ws) {
#pragma unroll
        for (int q = 0; q < 4; q++)
            ws_words[q] = q * 256 < amax_nblocks ? ((const uint4*)amax_ws)[q * 64 + (t & 63)] : make_uint4(0u, 0u, 0u, 0u);
    }

    Row8<DT> in[2][4];
    load_tile<DT, 2>(in, x, r0, c0, rows, cols, ld);

    // The scale: given -- or, for dynamic scaling, derived here from the per-workgroup maxima the amax kernel left in
    // amax_ws (every wave of every workgroup reduces the <= 1024 words itself; saves the one-block launch that would do
    // it once).  The words were requested before the tile and nothing here waits for anybody else, so the reduction
    // runs while the tile's loads are still in flight.  (A first version shared the work among the four waves through
    // LDS: its two barriers, in the middle of the block, cost more than the redundant loads do.)  Words past
    // amax_nblocks are leftovers of an earlier, larger call and are masked.  Same arithmetic as amax_finalize_kernel,
    // in the tensor's dtype.
    float scale;
    bool within;
    uint32_t m = 0;
    if (amax_ws) {
        uint32_t wm = 0;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int first = q * 256 + (t & 63) * 4;
            const uint32_t w[4] = {ws_words[q].x, ws_words[q].y, ws_words[q].z, ws_words[q].w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint32_t v = first + c < amax_nblocks ? w[c] : 0u;
                wm = wm > v ? wm : v;
            }
        }
        wm = wave_max_u32(wm);
        scale = amax_to_scale_dev(abs_bits_to_float(wm, DT), DT, FMT, DT == F8MI_FP16);
        if (bid == 0 && t == 0) *j.scale_out = scale;
        within = within_range<FMT>(abs_bits_to_float(wm, DT), scale);
    } else {
        scale = *j.scale_dev;
        m = absmax_tile<DT, 2>(in);
        within = __all(within_range<FMT>(abs_bits_to_float(m, DT), scale));
    }

    emit_tile<DT, PROD, FMT, 2>(in, tileT, scale, within, r0, c0, rows, cols, j.out, j.out_t, j.out_kb, j.out_t_kb);

    if constexpr (TAGGED) {
        // Every wave leaves its maximum in a word of its own; the workgroup that was started last collects them.
        m = wave_max_u32(m);
        if ((t & 63) == 0) publish_word(j.tagged, bid * (CAST_THREADS / 64) + (t >> 6), m);
        if (bid == nb - 1) {
            if (__builtin_expect(!collect_words<8>(j.tagged, nb * (CAST_THREADS / 64), m, red), 0)) m = collect_alone<DT>(j, red);
            if (t == 0) *amax_out = abs_bits_to_float(m, DT);
        }
    } else if (amax_out && j.amax_spread) {
        // Every wave folds its maximum (the bit pattern in the input's dtype) into one of SPREAD_WORDS words with an
        // atomic that returns nothing: no LDS, no barrier, no round trip to wait for, and a word sees about one atomic
        // per (tiles * 4 / SPREAD_WORDS) waves, spread over the whole run of the kernel.  cast_spread_finalize_kernel
        // turns the words into *amax_out.  (Measured per tensor of the benchmark, 128 MB .. 1.8 GB, against the cast
        // without amax: folding into *amax_out itself, one compare-and-atomic per workgroup at its end as below, +6 ..
        // +20 us -- the workgroup holds its LDS and wave slots for the round trip of that last read; this + 0 .. 2 us,
        // plus 4 us for the finalize launch.)
        m = wave_max_u32(m);
        if ((t & 63) == 0 && m)
            (void)__hip_atomic_fetch_max(&j.amax_spread[(bid * (CAST_THREADS / 64) + (t >> 6)) & (SPREAD_WORDS - 1)], m,
                                         __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    } else if (amax_out) {
        m = wave_max_u32(m);
        const int wave = t >> 6, lane = t & 63;
        if (lane == 0) red[wave] = m;
        __syncthreads();
        if (wave == 0) {
            uint32_t v = lane < CAST_THREADS / 64 ? red[lane] : 0u;
            m = wave_max_u32(v);
        }
        publish_amax_cast(m, amax_out, DT);
    }
}

template <int DT, int PROD, int FMT, bool TAGGED>
__global__ __launch_bounds__(CAST_THREADS) void cast_kernel(CastJob j) {
    __shared__ uint32_t tileT[CAST_TILE * CAST_TILE / 4];  // [column][row/4] dwords, swizzled
    __shared__ uint32_t red[CAST_THREADS / 64];
    cast_body<DT, PROD, FMT, TAGGED>(j, blockIdx.x, gridDim.x, tileT, red);
}

// Two tensors in one launch, the first nb_a workgroups for the first.  TAGGED: delayed scaling, the product in fp32.
template <int DTA, int DTB, int FMT, bool TAGGED>
__global__ __launch_bounds__(CAST_THREADS) void cast_pair_kernel(CastJob a, CastJob b, uint32_t nb_a) {
    __shared__ uint32_t tileT[CAST_TILE * CAST_TILE / 4];
    __shared__ uint32_t red[CAST_THREADS / 64];
    if (blockIdx.x < nb_a) cast_body<DTA, TAGGED ? F8MI_FP32 : DTA, FMT, TAGGED>(a, blockIdx.x, nb_a, tileT, red);
    else cast_body<DTB, TAGGED ? F8MI_FP32 : DTB, FMT, TAGGED>(b, blockIdx.x - nb_a, gridDim.x - nb_a, tileT, red);
}

// Dynamic scaling of a small tensor in ONE launch: amax, scale and cast by a single workgroup that holds the whole
// tensor in registers (at most four items of eight elements per lane, loaded back to back).  Same arithmetic,
// element for element, as amax kernel + cast kernel; it exists because three or four launches cost more than
// the work when the tensor is a few rows of activations.
constexpr int SMALL_THREADS = 1024;
constexpr int SMALL_ITEMS_PER_THREAD = 4;
constexpr int64_t SMALL_MAX_ITEMS = (int64_t)SMALL_THREADS * SMALL_ITEMS_PER_THREAD;  // 32 K elements: 64 KB of bf16

template <int DT, int FMT>
__global__ __launch_bounds__(SMALL_THREADS) void cast_dynamic_small_kernel(const void* __restrict__ x, int64_t rows, int64_t cols,
                                                                           int64_t ld, float* __restrict__ scale_out,
                                                                           uint8_t* __restrict__ out, uint8_t* __restrict__ out_t,
                                                                           int out_kb, int out_t_kb) {
    __shared__ uint32_t red[SMALL_THREADS / 64];
    __shared__ uint32_t amax_bits;
    const int t = threadIdx.x;
    const int64_t groups = (cols + 7) / 8, items = rows * groups;  // an item: eight consecutive elements of a row
    Row8<DT> r[SMALL_ITEMS_PER_THREAD];
    uint32_t m = 0;
#pragma unroll
    for (int u = 0; u < SMALL_ITEMS_PER_THREAD; u++) {
        const int64_t it = t + (int64_t)u * SMALL_THREADS;
        // past the last item: row == rows, which load_row8 reads as zeros
        load_row8<DT>(r[u], x, it < items ? it / groups : rows, (it % groups) * 8, rows, cols, ld);
    }
#pragma unroll
    for (int u = 0; u < SMALL_ITEMS_PER_THREAD; u++) m = absmax_row<DT>(r[u], m);
    m = wave_max_u32(absmax_done<DT>(m));
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    if (t < 64) {
        uint32_t v = t < SMALL_THREADS / 64 ? red[t] : 0u;
        v = wave_max_u32(v);
        if (t == 0) amax_bits = v;
    }
    __syncthreads();
    // the scale in the tensor's own dtype, as tensor_to_scale computes it (fp16 tensors: clamped to 65504)
    const float amax = abs_bits_to_float(amax_bits, DT), scale = amax_to_scale_dev(amax, DT, FMT, DT == F8MI_FP16);
    if (t == 0) *scale_out = scale;
    const bool within = within_range<FMT>(amax, scale);
#pragma unroll
    for (int u = 0; u < SMALL_ITEMS_PER_THREAD; u++) {
        const int64_t it = t + (int64_t)u * SMALL_THREADS;
        if (it >= items) continue;
        const int64_t row = it / groups, col = (it % groups) * 8;
        uint32_t lo, hi;
        if (within) cast_row8<DT, DT, FMT, true>(r[u], scale, lo, hi);
        else cast_row8<DT, DT, FMT, false>(r[u], scale, lo, hi);
        if (out) {
            uint8_t* p = out_kb ? out + ((col >> 6) * rows + row) * 64 + (col & 63) : out + row * cols + col;
            if (col + 8 <= cols) {
                store8_any(p, lo, hi);
            } else {
#pragma unroll
                for (int i = 0; i < 8; i++)
                    if (col + i < cols) p[i] = (uint8_t)((i < 4 ? lo >> (8 * i) : hi >> (8 * (i - 4))) & 0xffu);
            }
        }
        if (out_t) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int64_t c = col + i;
                if (c < cols) {
                    uint8_t* p = out_t_kb ? out_t + ((row >> 6) * cols + c) * 64 + (row & 63) : out_t + c * rows + row;
                    *p = (uint8_t)((i < 4 ? lo >> (8 * i) : hi >> (8 * (i - 4))) & 0xffu);
                }
            }
        }
    }
}

template <int DT>
static int launch_cast_small(int fmt, hipStream_t stream, const void* x, int64_t rows, int64_t cols, int64_t ld,
                             float* scale_dev, uint8_t* out, uint8_t* out_t, int out_kb, int out_t_kb) {
    const dim3 g(1), b(SMALL_THREADS);
    if (fmt == F8MI_E4M3FN) hipLaunchKernelGGL((cast_dynamic_small_kernel<DT, F8MI_E4M3FN>), g, b, 0, stream, x, rows, cols, ld, scale_dev, out, out_t, out_kb, out_t_kb);
    else hipLaunchKernelGGL((cast_dynamic_small_kernel<DT, F8MI_E5M2>), g, b, 0, stream, x, rows, cols, ld, scale_dev, out, out_t, out_kb, out_t_kb);
    return check_hip(hipGetLastError(), "cast (dynamic, one workgroup) kernel launch");
}

// Dynamic scaling of a few rows of activations, one copy, in ONE launch: every workgroup finds the maximum of the whole
// tensor itself (the tensor sits in every XCD's L2 after the first workgroup there has read it), then casts its own 8 K
// elements, one item of eight per lane, requested ahead of the scan.  Latency-bound: what it saves is the launch of the
// amax pass and the gap behind it; what it costs is the scan at the rate of one CU, which grows with the tensor while the two
// kernels' time does not.  Same arithmetic, element for element, as those: the same bits.
//
// us a call, back to back, two kernels / this one: bf16, 16 x 4096: 6.8 / 3.5, 32 x 4096: 7.3 / 4.4, 64 x 4096 (512 KB): 7.3 / 6.3,
// 64 x 8192: 7.4 / 9.9; fp32, 16 x 4096: 6.8 / 4.3, 32 x 4096 (512 KB): 6.9 / 6.1, 16 x 14336 (896 KB): 6.9 / 8.7.  In place, between
// products with a cold weight of 4096 rows, cast and product together: bf16, 16 x 4096: 15.0 / 10.6, 64 x 4096 (512 KB): 20.7 / 19.1, 32 x
// 8192 (512 KB): 22.8 / 21.6, 16 x 14336 (448 KB): 23.5 / 22.1; fp32, 16 x 4096: 15.3 / 12.1, 16 x 8192 (512 KB): 18.8 / 18.3.  Hence the line.
constexpr int FLAT_THREADS = 1024;
constexpr int FLAT_UNROLL = 8;  // 16-byte loads in flight per lane of the scan
constexpr int64_t FLAT_MAX_BYTES = 512 << 10;
// Past this many bytes the kernel that reads the tensor once (cast_dynamic_resident_kernel) is faster, where the stream has its words:
// us, this / that: 32 x 4096 (256 KB): 5.5 / 5.8, 48 x 4096: 6.3 / 5.9, 16 x 14336 (448 KB): 7.2 / 6.3, 64 x 4096: 7.3 / 5.9.  Its tiles
// have 64 rows, so that few rows are many tiles of mostly nothing: bf16, 8 rows 320 KB 6.44 / 7.31, 448 KB 7.55 / 7.57; 10 rows 6.44 / 6.46, 384 KB 6.66 /
// 7.11; 12 rows 320 KB 6.52 / 6.38, 384 KB 6.62 / 6.45, 512 KB 7.77 / 7.30; fp32, 4 rows 320 KB 6.34 / 7.20, 8 rows 6.37 / 6.22, 12 rows 6.46 / 6.01.
constexpr int64_t FLAT_BEST_BYTES = 320 << 10;
constexpr int64_t FLAT_BEST_ROWS = 12;

template <int DT, int FMT>
__global__ __launch_bounds__(FLAT_THREADS) void cast_dynamic_flat_kernel(const uint8_t* __restrict__ x, uint32_t rows, uint32_t cols,
                                                                         uint32_t items, float* __restrict__ scale_out,
                                                                         uint8_t* __restrict__ out, int out_kb) {
    constexpr uint32_t VEC_PER_ITEM = DT == F8MI_FP32 ? 2 : 1;
    __shared__ uint32_t red[FLAT_THREADS / 64];
    const uint32_t t = threadIdx.x, own = blockIdx.x * FLAT_THREADS + t, last = items * VEC_PER_ITEM - 1;
    auto load = [&](uint32_t i) __attribute__((always_inline)) { return *(const u32x4_any*)(x + (size_t)min(i, last) * 16); };
    Row8<DT> r;  // past the last item: the last vector again, not stored
#pragma unroll
    for (uint32_t h = 0; h < VEC_PER_ITEM; h++) {
        const u32x4 q = load(own * VEC_PER_ITEM + h);
        r.w[4 * h] = q.x; r.w[4 * h + 1] = q.y; r.w[4 * h + 2] = q.z; r.w[4 * h + 3] = q.w;
    }
    uint32_t m = 0;
    for (uint32_t i = t; i <= last; i += FLAT_UNROLL * FLAT_THREADS) {
        u32x4 v[FLAT_UNROLL];
#pragma unroll
        for (int u = 0; u < FLAT_UNROLL; u++) v[u] = load(i + u * FLAT_THREADS);
#pragma unroll
        for (int u = 0; u < FLAT_UNROLL; u++) {
            const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int c = 0; c < 4; c++) {
                if constexpr (DT == F8MI_FP32) m = max(m, w[c] & 0x7fffffffu);
                else m = absmax16x2(w[c], m);
            }
        }
    }
    m = wave_max_u32(absmax_done<DT>(m));
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    m = red[0];
#pragma unroll
    for (int i = 1; i < FLAT_THREADS / 64; i++) m = max(m, red[i]);
    const float amax = abs_bits_to_float(m, DT), scale = amax_to_scale_dev(amax, DT, FMT, DT == F8MI_FP16);
    if (own == 0) *scale_out = scale;
    if (own >= items) return;
    uint32_t lo, hi;
    if (within_range<FMT>(amax, scale)) cast_row8<DT, DT, FMT, true>(r, scale, lo, hi);
    else cast_row8<DT, DT, FMT, false>(r, scale, lo, hi);
    size_t at = (size_t)own * 8;
    if (out_kb) {
        const uint32_t row = own / (cols / 8), col = (own - row * (cols / 8)) * 8;
        at = ((size_t)(col >> 6) * rows + row) * 64 + (col & 63);
    }
    store8_any(out + at, lo, hi);
}

template <int DT>
static int launch_cast_flat(int fmt, hipStream_t stream, const void* x, int64_t rows, int64_t cols, float* scale_dev, uint8_t* out, int out_kb) {
    const uint32_t items = (uint32_t)(rows * cols / 8);
    const dim3 g((items + FLAT_THREADS - 1) / FLAT_THREADS), b(FLAT_THREADS);
    if (fmt == F8MI_E4M3FN) hipLaunchKernelGGL((cast_dynamic_flat_kernel<DT, F8MI_E4M3FN>), g, b, 0, stream, (const uint8_t*)x, (uint32_t)rows, (uint32_t)cols, items, scale_dev, out, out_kb);
    else hipLaunchKernelGGL((cast_dynamic_flat_kernel<DT, F8MI_E5M2>), g, b, 0, stream, (const uint8_t*)x, (uint32_t)rows, (uint32_t)cols, items, scale_dev, out, out_kb);
    return check_hip(hipGetLastError(), "cast (dynamic, few rows) kernel launch");
}

// Dynamic scaling of a tensor that the chip can hold, any layout and both copies, in ONE launch that reads it once: every
// workgroup loads its tile (64 H rows x 128 columns) into registers, publishes the tile's maximum, collects everybody's and casts
// what it holds.  The two kernels it replaces read the tensor twice and pay a launch and a ramp more.
//
// Alone on the chip all workgroups are there at once (see resident_tile_rows).  Beside other streams' kernels they may not be: whoever
// waits for too long reads the missing tiles itself (see collect_late).  The kernel keeps nothing for that path in registers.
//
// us a call, back to back, inputs cold, amax and cast / this one: one copy, bf16, 512 x 1024: 8.8 / 6.4, 2048 x 2048: 10.6 / 9.0, 2726 x 934
// (padded): 16.1 / 10.7, 2048 x 4096: 14.3 / 11.5, 4096 x 4096: 20.5 / 17.6; both copies, 4096 x 4096: 21.8 / 19.3; fp32,
// 512 x 1024: 9.9 / 6.4, 4096 x 4096: 30.7 / 24.3.  (Twice as many tiles, all that eight workgroups a CU hold: 8192 x 4096 34.7 / 31.3 -- but then
// any other kernel on the chip makes all of them late: not taken.)  Inside a launch of 4096 x 4096 bf16 (1024 workgroups): the last tile has arrived after 9.5
// us, everybody has everybody's maximum after 11.3 (2 us is what a word takes to memory and back, 512 x 1024 waits as long), the
// last byte is stored after 15.  Loads in smaller batches, other tile shapes and linear tile orders all took the same or longer.
constexpr int RESIDENT_TILES = 1024;  // workgroups at most
// of two 16-bit tensors together, six workgroups a CU: see pair_tile_rows
constexpr int RESIDENT_PAIR_TILES = 1536;

template <int DT, int FMT, int H>
__device__ __forceinline__ void resident_body(const CastJob& j, uint32_t bid, uint32_t nb, uint32_t* tileT, uint32_t* red) {
    const int t = threadIdx.x;
    int ty, tx;
    cast_tile_of(bid, nb, j.tiles_x, j.tiles_y, ty, tx);
    const int64_t r0 = (int64_t)ty * (64 * H), c0 = (int64_t)tx * CAST_TILE;
    Row8<DT> in[H][4];
    load_tile<DT, H>(in, j.x, r0, c0, j.rows, j.cols, j.ld);
    uint32_t m = wave_max_u32(absmax_tile<DT, H>(in));
    if ((t & 63) == 0) red[t >> 6] = m;
    __syncthreads();
    if (t == 0) publish_word(j.tagged, bid, max(max(red[0], red[1]), max(red[2], red[3])));
    if (__builtin_expect(!collect_words<1>(j.tagged, nb, m, red + CAST_THREADS / 64), 0)) {
        m = collect_late<DT, H>(j, bid, nb, red);
        // The tile again: held meanwhile, it or its addresses would cost every launch registers, and a CU a workgroup.
        int64_t again = r0;
        asm volatile("" : "+s"(again));
        load_tile<DT, H>(in, j.x, again, c0, j.rows, j.cols, j.ld);
    }
    const float amax = abs_bits_to_float(m, DT), scale = amax_to_scale_dev(amax, DT, FMT, DT == F8MI_FP16);
    if (bid == 0 && t == 0) *j.scale_out = scale;
    emit_tile<DT, DT, FMT, H>(in, tileT, scale, within_range<FMT>(amax, scale), r0, c0, j.rows, j.cols, j.out, j.out_t, j.out_kb, j.out_t_kb);
}

template <int DT, int FMT, int H>
__global__ __launch_bounds__(CAST_THREADS) void cast_dynamic_resident_kernel(CastJob j) {
    __shared__ uint32_t tileT[32 * 64 * H];
    __shared__ uint32_t red[2 * CAST_THREADS / 64];
    resident_body<DT, FMT, H>(j, blockIdx.x, gridDim.x, tileT, red);
}

// Two tensors that fit together; each finds its own maximum.
template <int DTA, int DTB, int FMT, int H>
__global__ __launch_bounds__(CAST_THREADS) void cast_dynamic_resident_pair_kernel(CastJob a, CastJob b, uint32_t nb_a) {
    __shared__ uint32_t tileT[32 * 64 * H];
    __shared__ uint32_t red[2 * CAST_THREADS / 64];
    if (blockIdx.x < nb_a) resident_body<DTA, FMT, H>(a, blockIdx.x, nb_a, tileT, red);
    else resident_body<DTB, FMT, H>(b, blockIdx.x - nb_a, gridDim.x - nb_a, tileT, red);
}

constexpr int STATIC_MAX_DEVICES = 64;

// Device address of a device array of this library on the current device, looked up once per device and kept (nullptr + error
// message on failure).  Two threads racing here store the same value.
template <typename T>
static T* device_array(const void* symbol, std::atomic<T*> (&known)[STATIC_MAX_DEVICES], const char* what) {
    int dev = -1;
    if (check_hip(hipGetDevice(&dev), "hipGetDevice")) return nullptr;
    if (dev < 0 || dev >= STATIC_MAX_DEVICES) { set_error("%s: device index %d, at most %d devices", what, dev, STATIC_MAX_DEVICES); return nullptr; }
    if (T* p = known[dev].load(std::memory_order_acquire)) return p;
    void* addr = nullptr;
    if (check_hip(hipGetSymbolAddress(&addr, symbol), what)) return nullptr;
    if (!addr) { set_error("%s: no address on device %d", what, dev); return nullptr; }
    known[dev].store((T*)addr, std::memory_order_release);
    return (T*)addr;
}

// The words of the exchanges: a set for each of the last EXCHANGE_STREAMS streams to use one for the first time, so that launches which
// may run at the same time do not share any (sharing would be slow, not wrong).  A further stream takes over the set that was given
// out first, whose stream may be gone; if it is not, it gets another with its next launch.  Streams that are being captured have none: a captured launch would
// use its tag again on every replay.  A stream handle that comes back for a new stream finds the old one's set: its work is done.
constexpr int EXCHANGE_STREAMS = 64;
constexpr int EXCHANGE_WORDS = 8192;
static __device__ __align__(256) uint64_t exchange_words[EXCHANGE_STREAMS][EXCHANGE_WORDS];
static std::atomic<uint64_t*> g_exchange_words[STATIC_MAX_DEVICES];
static std::atomic<uintptr_t> g_exchange_streams[STATIC_MAX_DEVICES][EXCHANGE_STREAMS];
static std::atomic<uint32_t> g_exchange_last[STATIC_MAX_DEVICES][EXCHANGE_STREAMS];  // tag of the set's last launch
static std::atomic<uint32_t> g_exchange_given[STATIC_MAX_DEVICES];
static std::atomic<uint32_t> g_exchange_tag{0};
constexpr uint32_t EXCHANGE_LATELY = 64;  // launches

static int exchange_set(int dev, hipStream_t stream) {
    static thread_local char own;  // one handle stands for every thread's own stream
    const uintptr_t key = stream == hipStreamPerThread ? (uintptr_t)&own : (uintptr_t)stream + 1;  // the default stream is a null handle
    for (int i = 0; i < EXCHANGE_STREAMS; i++)
        if (g_exchange_streams[dev][i].load(std::memory_order_relaxed) == key) return i;
    const int i = (int)(g_exchange_given[dev].fetch_add(1, std::memory_order_relaxed) % EXCHANGE_STREAMS);
    g_exchange_streams[dev][i].store(key, std::memory_order_relaxed);
    return i;
}

// Words and a tag for one launch on `stream`; words null: none to be had.  An error code if the runtime reports one.
// streams: how many streams of the device, this one among them, had one of the last EXCHANGE_LATELY launches.
static int begin_exchange(hipStream_t stream, uint32_t wait_ticks, TaggedWords& e, int* streams = nullptr) {
    e = TaggedWords{nullptr, 0, wait_ticks};
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &capture) != hipSuccess) {  // of the default stream, say, while a blocking one is captured: launches are taken
        (void)hipGetLastError();
        return F8MI_OK;
    }
    if (capture != hipStreamCaptureStatusNone) return F8MI_OK;
    int dev = 0;
    if (check_hip(hipGetDevice(&dev), "hipGetDevice")) return F8MI_ERR_HIP;
    uint64_t* base = device_array(HIP_SYMBOL(exchange_words), g_exchange_words, "exchange_words");
    if (!base) return F8MI_ERR_HIP;
    const int set = exchange_set(dev, stream);
    e.words = base + (size_t)set * EXCHANGE_WORDS;
    e.tag = g_exchange_tag.fetch_add(1, std::memory_order_relaxed) + 1;
    if (!e.tag) e.tag = g_exchange_tag.fetch_add(1, std::memory_order_relaxed) + 1;  // 0 is what the words start with
    g_exchange_last[dev][set].store(e.tag, std::memory_order_relaxed);
    if (streams) {
        *streams = 0;
        for (const auto& last : g_exchange_last[dev]) {
            const uint32_t tag = last.load(std::memory_order_relaxed);
            *streams += tag && e.tag - tag < EXCHANGE_LATELY;  // (another thread's may be newer: not counted)
        }
    }
    return F8MI_OK;
}

// where a dynamic-scaling cast takes its scale from (see cast_layout_impl)
struct AmaxSource {
    const uint32_t* ws;
    int nblocks;
    float* scale_out;
    uint32_t* spread;  // delayed scaling: the zeroed words the fused amax is folded into (null: straight into *amax_dev)
    TaggedWords tagged;  // delayed scaling in one launch: instead of those
};

__global__ void cast_zero_amax_kernel(float* amax_out) {
    if (threadIdx.x == 0) *amax_out = 0.0f;
}

// Second half of the fused amax with a workspace: the maximum of the SPREAD_WORDS words becomes *amax_out (widened to
// fp32) and every word goes back to zero, which is the state the next call expects.  One workgroup.
__global__ __launch_bounds__(SPREAD_WORDS) void cast_spread_finalize_kernel(uint32_t* __restrict__ spread, float* __restrict__ amax_out, int in_dt) {
    __shared__ uint32_t red[SPREAD_WORDS / 64];
    uint32_t m = spread[threadIdx.x];
    if (m) spread[threadIdx.x] = 0u;
    m = wave_max_u32(m);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x < 64) {
        m = wave_max_u32(threadIdx.x < SPREAD_WORDS / 64 ? red[threadIdx.x] : 0u);
        if (threadIdx.x == 0) *amax_out = abs_bits_to_float(m, in_dt);
    }
}

// LDS that a cast asks for without using it, to be held to six workgroups a CU instead of the eight (fp32: four instead of five) that its
// registers allow, where its tiles number two rounds of them or more.  More of them at a time write more rows and columns at a time than
// the memory takes at full rate.  us, eight / six, bf16: 8192 x 4096 22.7 / 23.3, 12288 x 4096 32.0 / 32.0, 8192 x 14336 71.7 / 69.3, 28672 x 8192 140 /
// 138; with both copies 29.7 / 30.1, 42.7 / 42.1, 97.7 / 95.2, 187 / 182; fp32 with both, five / four: 8192 x 4096 43.8 / 43.4, 28672 x 8192 290 / 285.
constexpr unsigned UNUSED_LDS_16 = 10 << 10, UNUSED_LDS_32 = 20 << 10;
static unsigned unused_lds(int in_dtype, int64_t tiles) {
    const bool wide = in_dtype == F8MI_FP32;
    return tiles >= (wide ? 8 : 12) * (int64_t)cu_count() ? (wide ? UNUSED_LDS_32 : UNUSED_LDS_16) : 0u;
}
template <int DT, int PROD, int FMT>
static int launch_cast2(dim3 g, hipStream_t stream, const CastJob& j) {
    if constexpr (PROD == F8MI_FP32) {  // what delayed scaling computes in
        if (j.tagged.words) {
            hipLaunchKernelGGL((cast_kernel<DT, PROD, FMT, true>), g, dim3(CAST_THREADS), 0, stream, j);
            return check_hip(hipGetLastError(), "cast kernel launch");
        }
    }
    hipLaunchKernelGGL((cast_kernel<DT, PROD, FMT, false>), g, dim3(CAST_THREADS), unused_lds(DT, g.x), stream, j);
    return check_hip(hipGetLastError(), "cast kernel launch");
}

template <int DT, int PROD>
static int launch_cast1(int fmt, dim3 g, hipStream_t stream, const CastJob& j) {
    if (fmt == F8MI_E4M3FN) return launch_cast2<DT, PROD, F8MI_E4M3FN>(g, stream, j);
    return launch_cast2<DT, PROD, F8MI_E5M2>(g, stream, j);
}

static int check_cast_layouts(int64_t rows, int64_t cols, const void* out, int out_layout, const void* out_t, int out_t_layout) {
    if (out_layout < F8MI_LAYOUT_ROWMAJOR || out_layout > F8MI_LAYOUT_KBLOCK64_PAD128 || out_t_layout < F8MI_LAYOUT_ROWMAJOR || out_t_layout > F8MI_LAYOUT_KBLOCK64_PAD128) { set_error("f8mi_cast: unknown layout code"); return F8MI_ERR_INVALID_ARG; }
    if (out && out_layout == F8MI_LAYOUT_KBLOCK64 && cols % 64 != 0) { set_error("f8mi_cast: k-blocked `out` needs cols %% 64 == 0 (cols=%lld); F8MI_LAYOUT_KBLOCK64_PAD128 takes any", (long long)cols); return F8MI_ERR_UNSUPPORTED; }
    if (out_t && out_t_layout == F8MI_LAYOUT_KBLOCK64 && rows % 64 != 0) { set_error("f8mi_cast: k-blocked `out_t` needs rows %% 64 == 0 (rows=%lld); F8MI_LAYOUT_KBLOCK64_PAD128 takes any", (long long)rows); return F8MI_ERR_UNSUPPORTED; }
    return F8MI_OK;
}

// Validates and launches the cast.  `src.ws` null: the scale is read from scale_dev (f8mi_cast_layout).  Not null
// (dynamic scaling, product in the input's dtype): the kernel derives the scale from the src.nblocks per-workgroup
// maxima in src.ws and workgroup 0 stores it to src.scale_out.
static int cast_layout_impl(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, const float* scale_dev,
                            int product_dtype, int fp8_fmt, uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout,
                            float* amax_dev, hipStream_t stream, const AmaxSource& src) {
    if (const int rc = check_cast_layouts(rows, cols, out, out_layout, out_t, out_t_layout)) return rc;
    // the kernel takes the layout codes as they are (0: row-major, otherwise k-blocked; PAD128: whole tiles are written)
    const int out_kb = out ? out_layout : F8MI_LAYOUT_ROWMAJOR, out_t_kb = out_t ? out_t_layout : F8MI_LAYOUT_ROWMAJOR;
    // ld == 0: every row reads the same `cols` elements (the kernels address row * ld + col)
    if (rows < 0 || cols < 0 || (ld < cols && ld != 0)) { set_error("f8mi_cast: bad shape rows=%lld cols=%lld ld=%lld", (long long)rows, (long long)cols, (long long)ld); return F8MI_ERR_INVALID_ARG; }
    if (in_dtype < 0 || in_dtype > 2 || fp8_fmt < 0 || fp8_fmt > 1) { set_error("f8mi_cast: unknown dtype/format code"); return F8MI_ERR_INVALID_ARG; }
    if (product_dtype != in_dtype && product_dtype != F8MI_FP32) { set_error("f8mi_cast: product_dtype must be the input dtype or fp32"); return F8MI_ERR_INVALID_ARG; }
    if (!scale_dev && !src.ws) { set_error("f8mi_cast: null scale"); return F8MI_ERR_INVALID_ARG; }
    if (!out && !out_t && !amax_dev) { set_error("f8mi_cast: no output requested"); return F8MI_ERR_INVALID_ARG; }
    if (rows == 0 || cols == 0) {
        if (amax_dev) {
            hipLaunchKernelGGL(cast_zero_amax_kernel, dim3(1), dim3(64), 0, stream, amax_dev);
            return check_hip(hipGetLastError(), "cast_zero_amax_kernel");
        }
        return F8MI_OK;
    }
    if (!x) { set_error("f8mi_cast: null tensor"); return F8MI_ERR_INVALID_ARG; }
    const int64_t ty = (rows + CAST_TILE - 1) / CAST_TILE, tx = (cols + CAST_TILE - 1) / CAST_TILE;
    if (tx * ty > 0x7fffffffLL) { set_error("f8mi_cast: more than 2^31 tiles"); return F8MI_ERR_UNSUPPORTED; }
    dim3 g((unsigned)(tx * ty));
    const uint32_t tiles_x = (uint32_t)tx, tiles_y = (uint32_t)ty;
    const CastJob j{x, rows, cols, ld, out, out_t, tiles_x, tiles_y, out_kb, out_t_kb, scale_dev, src.scale_out, src.ws, src.nblocks, amax_dev, src.spread, src.tagged};
    const size_t esz = in_dtype == F8MI_FP32 ? 4 : 2;
    const double n = (double)rows * (double)cols;
    // every launch of this call: the cast and what a fused amax adds before or after it
    ProfScope prof(F8MI_K_CAST, (ld == 0 ? (double)cols : n) * esz + n * ((out ? 1 : 0) + (out_t ? 1 : 0)), stream);
    if (amax_dev && !src.spread && !src.tagged.words) {
        hipLaunchKernelGGL(cast_zero_amax_kernel, dim3(1), dim3(64), 0, stream, amax_dev);
        if (int rc = check_hip(hipGetLastError(), "cast_zero_amax_kernel")) return rc;
    }
    int rc;
    if (in_dtype == F8MI_BF16) {
        if (product_dtype == F8MI_BF16) rc = launch_cast1<F8MI_BF16, F8MI_BF16>(fp8_fmt, g, stream, j);
        else rc = launch_cast1<F8MI_BF16, F8MI_FP32>(fp8_fmt, g, stream, j);
    } else if (in_dtype == F8MI_FP16) {
        if (product_dtype == F8MI_FP16) rc = launch_cast1<F8MI_FP16, F8MI_FP16>(fp8_fmt, g, stream, j);
        else rc = launch_cast1<F8MI_FP16, F8MI_FP32>(fp8_fmt, g, stream, j);
    } else {
        rc = launch_cast1<F8MI_FP32, F8MI_FP32>(fp8_fmt, g, stream, j);
    }
    if (rc || !(amax_dev && src.spread)) return rc;
    hipLaunchKernelGGL(cast_spread_finalize_kernel, dim3(1), dim3(SPREAD_WORDS), 0, stream, src.spread, amax_dev, in_dtype);
    return check_hip(hipGetLastError(), "cast_spread_finalize_kernel");
}

}  // namespace f8mi

using namespace f8mi;

extern "C" int f8mi_cast_layout(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype,
                                const float* scale_dev, int product_dtype, int fp8_fmt, uint8_t* out, int out_layout,
                                uint8_t* out_t, int out_t_layout, float* amax_dev, void* stream) {
    return cast_layout_impl(x, rows, cols, ld, in_dtype, scale_dev, product_dtype, fp8_fmt, out, out_layout, out_t, out_t_layout, amax_dev,
                            (hipStream_t)stream, AmaxSource{});
}

extern "C" int f8mi_cast(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, const float* scale_dev,
                         int product_dtype, int fp8_fmt, uint8_t* out, uint8_t* out_t, float* amax_dev,
                         void* workspace, void* stream) {
    (void)workspace;
    return f8mi_cast_layout(x, rows, cols, ld, in_dtype, scale_dev, product_dtype, fp8_fmt, out, F8MI_LAYOUT_ROWMAJOR, out_t,
                            F8MI_LAYOUT_ROWMAJOR, amax_dev, stream);
}

extern "C" size_t f8mi_delayed_workspace_bytes(void) { return SPREAD_WORDS * sizeof(uint32_t); }

namespace f8mi {
// Host threads that share a workspace (and with it a stream) queue the cast and its finalize launch one pair at a time: with the
// finalize of one between the cast and the finalize of another, the first would take, and clear, both maxima.  The workspaces of
// different streams mostly find different locks; none is held for longer than two launches take to queue.
static std::mutex& delayed_lock(const void* workspace) {
    static std::mutex locks[64];
    return locks[((uintptr_t)workspace >> 12) % 64];
}

// The delayed cast in one launch: a word for every wave.
static bool one_launch_delayed(int64_t rows, int64_t cols) {
    const int64_t tx = (cols + CAST_TILE - 1) / CAST_TILE, ty = (rows + CAST_TILE - 1) / CAST_TILE, most = EXCHANGE_WORDS / (CAST_THREADS / 64);
    return tx <= most && ty <= most && tx * ty <= most;
}
}  // namespace f8mi

// F8MI_ERR_UNSUPPORTED, and nothing queued: not in one launch.
static int cast_delayed_one_launch(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, const float* scale_dev, int fp8_fmt, uint8_t* out,
                                   int out_layout, uint8_t* out_t, int out_t_layout, float* amax_dev, uint32_t wait_ticks, hipStream_t stream) {
    if (rows <= 0 || cols <= 0 || !one_launch_delayed(rows, cols)) return F8MI_ERR_UNSUPPORTED;
    AmaxSource src{};
    if (const int rc = begin_exchange(stream, wait_ticks, src.tagged)) return rc;
    if (!src.tagged.words) return F8MI_ERR_UNSUPPORTED;
    return cast_layout_impl(x, rows, cols, ld, in_dtype, scale_dev, F8MI_FP32, fp8_fmt, out, out_layout, out_t, out_t_layout, amax_dev, stream, src);
}

extern "C" int f8mi_cast_delayed(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, const float* scale_dev, int fp8_fmt,
                                 uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout, float* amax_dev, void* workspace,
                                 void* stream) {
    if (!amax_dev) { set_error("f8mi_cast_delayed: null amax"); return F8MI_ERR_INVALID_ARG; }
    if (!workspace || (uintptr_t)workspace % 4 != 0) { set_error("f8mi_cast_delayed: null or misaligned workspace"); return F8MI_ERR_INVALID_ARG; }
    {
        const int rc = cast_delayed_one_launch(x, rows, cols, ld, in_dtype, scale_dev, fp8_fmt, out, out_layout, out_t, out_t_layout, amax_dev,
                                               EXCHANGE_WAIT_TICKS_LAST, (hipStream_t)stream);
        // (a cast that is refused for its layouts is refused again below, with the same message)
        if (rc != F8MI_ERR_UNSUPPORTED) return rc;
    }
    AmaxSource src{};
    src.spread = (uint32_t*)workspace;
    const std::lock_guard<std::mutex> guard(f8mi::delayed_lock(workspace));
    return cast_layout_impl(x, rows, cols, ld, in_dtype, scale_dev, F8MI_FP32, fp8_fmt, out, out_layout, out_t, out_t_layout, amax_dev,
                            (hipStream_t)stream, src);
}

namespace f8mi {

// Rows of the tiles that the one-launch cast gives a tensor, 0: it does not take it.  At most four workgroups a CU (RESIDENT_TILES on
// 256) of the eight that it holds, five of 128 rows of fp32: a launch that is alone has them all there at once, with room for another
// beside it (fp32: for a small one).
static int resident_tile_rows(int64_t rows, int64_t cols) {
    const int64_t tx = (cols + CAST_TILE - 1) / CAST_TILE, ty = (rows + CAST_TILE - 1) / CAST_TILE, most = std::min(RESIDENT_TILES, 4 * cu_count());
    if (ty > most || tx > most) return 0;
    // tiles of 64 rows while they number at most two a CU: more workgroups share a small tensor (512 x 1024: 7.6 -> 6.6 us); beyond that
    // they only add words to collect (2048 x 4096 as 512 or 1024 tiles: 12.2 / 12.5)
    return 2 * tx * ty <= most / 2 ? 64 : tx * ty <= most ? 128 : 0;
}

template <int DT, int FMT>
static int launch_cast_resident1(int tile_rows, dim3 g, hipStream_t stream, const CastJob& j) {
    if (tile_rows == 64) hipLaunchKernelGGL((cast_dynamic_resident_kernel<DT, FMT, 1>), g, dim3(CAST_THREADS), 0, stream, j);
    else hipLaunchKernelGGL((cast_dynamic_resident_kernel<DT, FMT, 2>), g, dim3(CAST_THREADS), 0, stream, j);
    return check_hip(hipGetLastError(), "cast (dynamic, resident) kernel launch");
}
template <int DT>
static int launch_cast_resident(int fmt, int tile_rows, dim3 g, hipStream_t stream, const CastJob& j) {
    if (fmt == F8MI_E4M3FN) return launch_cast_resident1<DT, F8MI_E4M3FN>(tile_rows, g, stream, j);
    return launch_cast_resident1<DT, F8MI_E5M2>(tile_rows, g, stream, j);
}

}  // namespace f8mi

extern "C" int f8mi_cast_dynamic_resident(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, int fp8_fmt, float* scale_dev,
                                          uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout, uint32_t wait_ticks, void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (rows <= 0 || cols <= 0 || (ld < cols && ld != 0) || in_dtype < 0 || in_dtype > 2 || fp8_fmt < 0 || fp8_fmt > 1) { set_error("f8mi_cast_dynamic_resident: bad shape or dtype/format code"); return F8MI_ERR_INVALID_ARG; }
    if (!x || !scale_dev || (!out && !out_t)) { set_error("f8mi_cast_dynamic_resident: null tensor or scale, or no output"); return F8MI_ERR_INVALID_ARG; }
    if (const int rc = check_cast_layouts(rows, cols, out, out_layout, out_t, out_t_layout)) return rc;
    const int tile_rows = resident_tile_rows(rows, cols);
    if (!tile_rows) { set_error("f8mi_cast_dynamic_resident: %lld x %lld is more than the chip holds", (long long)rows, (long long)cols); return F8MI_ERR_UNSUPPORTED; }
    TaggedWords tagged;
    if (const int rc = begin_exchange(stream, wait_ticks, tagged)) return rc;
    if (!tagged.words) { set_error("f8mi_cast_dynamic_resident: the stream is being captured"); return F8MI_ERR_UNSUPPORTED; }
    const int out_kb = out ? out_layout : F8MI_LAYOUT_ROWMAJOR, out_t_kb = out_t ? out_t_layout : F8MI_LAYOUT_ROWMAJOR;
    // whole 128 x 128 tiles, as the padded layouts are
    const uint32_t tiles_x = (uint32_t)((cols + CAST_TILE - 1) / CAST_TILE), tiles_y = (uint32_t)((rows + CAST_TILE - 1) / CAST_TILE) * (CAST_TILE / tile_rows);
    const dim3 g(tiles_x * tiles_y);
    const CastJob j{x, rows, cols, ld, out, out_t, tiles_x, tiles_y, out_kb, out_t_kb, nullptr, scale_dev, nullptr, 0, nullptr, nullptr, tagged};
    const size_t esz = in_dtype == F8MI_FP32 ? 4 : 2;
    const double n = (double)rows * (double)cols;
    ProfScope prof(F8MI_K_CAST, (ld == 0 ? (double)cols : n) * esz + n * ((out ? 1 : 0) + (out_t ? 1 : 0)), stream);
    if (in_dtype == F8MI_BF16) return launch_cast_resident<F8MI_BF16>(fp8_fmt, tile_rows, g, stream, j);
    if (in_dtype == F8MI_FP16) return launch_cast_resident<F8MI_FP16>(fp8_fmt, tile_rows, g, stream, j);
    return launch_cast_resident<F8MI_FP32>(fp8_fmt, tile_rows, g, stream, j);
}

extern "C" int f8mi_cast_dynamic(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, int fp8_fmt, float* scale_dev,
                                 uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout, void* workspace, void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (!scale_dev) { set_error("f8mi_cast_dynamic: null scale"); return F8MI_ERR_INVALID_ARG; }
    if (rows < 0 || cols < 0 || (ld < cols && ld != 0) || in_dtype < 0 || in_dtype > 2 || fp8_fmt < 0 || fp8_fmt > 1) { set_error("f8mi_cast_dynamic: bad shape or dtype/format code"); return F8MI_ERR_INVALID_ARG; }
    const size_t esz = in_dtype == F8MI_FP32 ? 4 : 2;
    const int64_t n = rows * cols;
    const bool padded = (out && out_layout == F8MI_LAYOUT_KBLOCK64_PAD128) || (out_t && out_t_layout == F8MI_LAYOUT_KBLOCK64_PAD128);  // the tile kernel writes the padding
    if (n > 0 && rows * ((cols + 7) / 8) <= SMALL_MAX_ITEMS && (out || out_t) && !padded) {
        if ((out_layout != F8MI_LAYOUT_ROWMAJOR && out_layout != F8MI_LAYOUT_KBLOCK64) || (out_t_layout != F8MI_LAYOUT_ROWMAJOR && out_t_layout != F8MI_LAYOUT_KBLOCK64)) { set_error("f8mi_cast_dynamic: unknown layout code"); return F8MI_ERR_INVALID_ARG; }
        if (out && out_layout == F8MI_LAYOUT_KBLOCK64 && cols % 64 != 0) { set_error("f8mi_cast_dynamic: k-blocked `out` needs cols %% 64 == 0 (cols=%lld)", (long long)cols); return F8MI_ERR_UNSUPPORTED; }
        if (out_t && out_t_layout == F8MI_LAYOUT_KBLOCK64 && rows % 64 != 0) { set_error("f8mi_cast_dynamic: k-blocked `out_t` needs rows %% 64 == 0 (rows=%lld)", (long long)rows); return F8MI_ERR_UNSUPPORTED; }
        if (!x) { set_error("f8mi_cast_dynamic: null tensor"); return F8MI_ERR_INVALID_ARG; }
        const int out_kb = out_layout == F8MI_LAYOUT_KBLOCK64, out_t_kb = out_t_layout == F8MI_LAYOUT_KBLOCK64;
        ProfScope prof(F8MI_K_CAST, (double)n * (esz + (out ? 1 : 0) + (out_t ? 1 : 0)), stream);
        if (in_dtype == F8MI_BF16) return launch_cast_small<F8MI_BF16>(fp8_fmt, stream, x, rows, cols, ld, scale_dev, out, out_t, out_kb, out_t_kb);
        if (in_dtype == F8MI_FP16) return launch_cast_small<F8MI_FP16>(fp8_fmt, stream, x, rows, cols, ld, scale_dev, out, out_t, out_kb, out_t_kb);
        return launch_cast_small<F8MI_FP32>(fp8_fmt, stream, x, rows, cols, ld, scale_dev, out, out_t, out_kb, out_t_kb);
    }
    if (n == 0 || (!out && !out_t))  // only the scale is wanted
        return f8mi_amax_scale(x, rows, cols, ld, in_dtype, fp8_fmt, in_dtype, in_dtype == F8MI_FP16, nullptr, scale_dev, workspace, stream_);
    if (!x || !workspace) { set_error("f8mi_cast_dynamic: null tensor or workspace"); return F8MI_ERR_INVALID_ARG; }
    if ((uintptr_t)workspace % 16 != 0) {  // the cast reads the workspace in 16-byte pieces: an odd one takes the two calls as they are
        int rc = f8mi_amax_scale(x, rows, cols, ld, in_dtype, fp8_fmt, in_dtype, in_dtype == F8MI_FP16, nullptr, scale_dev, workspace, stream_);
        if (rc) return rc;
        return f8mi_cast_layout(x, rows, cols, ld, in_dtype, scale_dev, in_dtype, fp8_fmt, out, out_layout, out_t, out_t_layout, nullptr, stream_);
    }
    const bool flat = out && !out_t && cols % 8 == 0 && (ld == cols || rows == 1) && n * (int64_t)esz <= FLAT_MAX_BYTES && out_t_layout >= F8MI_LAYOUT_ROWMAJOR &&
                      out_t_layout <= F8MI_LAYOUT_KBLOCK64_PAD128 && (out_layout == F8MI_LAYOUT_ROWMAJOR || (out_layout == F8MI_LAYOUT_KBLOCK64 && cols % 64 == 0));
    if (resident_tile_rows(rows, cols) && !(flat && (n * (int64_t)esz <= FLAT_BEST_BYTES || rows < FLAT_BEST_ROWS))) {
        const int rc = f8mi_cast_dynamic_resident(x, rows, cols, ld, in_dtype, fp8_fmt, scale_dev, out, out_layout, out_t, out_t_layout, EXCHANGE_WAIT_TICKS, stream_);
        if (rc != F8MI_ERR_UNSUPPORTED) return rc;
    }
    if (flat) {
        const int out_kb = out_layout == F8MI_LAYOUT_KBLOCK64;
        ProfScope prof(F8MI_K_CAST, (double)n * (esz + 1), stream);
        if (in_dtype == F8MI_BF16) return launch_cast_flat<F8MI_BF16>(fp8_fmt, stream, x, rows, cols, scale_dev, out, out_kb);
        if (in_dtype == F8MI_FP16) return launch_cast_flat<F8MI_FP16>(fp8_fmt, stream, x, rows, cols, scale_dev, out, out_kb);
        return launch_cast_flat<F8MI_FP32>(fp8_fmt, stream, x, rows, cols, scale_dev, out, out_kb);
    }
    // amax pass: per-workgroup maxima into the workspace; the cast's workgroups reduce them and derive the scale
    // themselves (no one-block finalize launch in between), workgroup 0 stores it to *scale_dev
    int nblocks = 0;
    {
        ProfScope prof(F8MI_K_AMAX, (double)(ld == 0 ? cols : n) * esz, stream);
        if (int rc = launch_amax_partials(x, rows, cols, ld, in_dtype, (uint32_t*)workspace, stream, &nblocks)) return rc;
    }
    return cast_layout_impl(x, rows, cols, ld, in_dtype, nullptr, in_dtype, fp8_fmt, out, out_layout, out_t, out_t_layout, nullptr, stream,
                            AmaxSource{(const uint32_t*)workspace, nblocks, scale_dev, nullptr, {}});
}

namespace f8mi {

// Two tensors, the operands of one product, in one launch: what it saves is the second one's launch, ramp and, between them, the
// tail of the first.  us, back to back, inputs cold, two calls / this, bf16, dynamic: 512 x 1024 and 1024 x 1024: 12.8 / 7.0; 2048 x 4096
// twice (1024 tiles, one launch): 23.3 / 18.8; 8192 x 4096 and 1024 x 4096 (two launches): 42.9 / 37.5, and 14336 x 4096: 88.2 / 83.6;
// delayed: 11.5 / 6.1, 18.2 / 13.5, 2048 x 4096 and 4096 x 4096 22.6 / 18.9; bf16 and fp32, dynamic, 512 x 1024 and 1024 x 1024: 13.2 / 7.5.
static int64_t tiles_of(const f8mi_cast_job& j) {
    const int64_t ty = (j.rows + CAST_TILE - 1) / CAST_TILE, tx = (j.cols + CAST_TILE - 1) / CAST_TILE;
    return ty > 0x7fffffff || tx > 0x7fffffff || tx * ty > 0x3fffffff ? 0x40000000 : tx * ty;
}
// Whether both are what the pair kernels take; anything else, wrong arguments among it, is left to the two calls.
static bool pair_ok(const f8mi_cast_job& a, const f8mi_cast_job& b) {
    for (const f8mi_cast_job* j : {&a, &b})
        if (j->rows <= 0 || j->cols <= 0 || (j->ld < j->cols && j->ld != 0) || !j->x || !j->scale_dev || (!j->out && !j->out_t) || j->in_dtype < 0 || j->in_dtype > 2 ||
            check_cast_layouts(j->rows, j->cols, j->out, j->out_layout, j->out_t, j->out_t_layout) || tiles_of(*j) >= 0x40000000)
            return false;
    return a.in_dtype == b.in_dtype || b.in_dtype == F8MI_FP32;
}
static int64_t job_read(const f8mi_cast_job& j) { return j.rows * j.cols * (j.in_dtype == F8MI_FP32 ? 4 : 2); }
// The maxima of both in one launch and their casts in another: where both take two launches by themselves, and where the one that
// takes only one is small: it is read twice that way (8192 x 4096 with 1024 x 4096: 42.9 / 37.5 us, with 4096 x 4096 fp32: 59.5 / 61.7).
static bool two_launches_pay(const f8mi_cast_job& a, const f8mi_cast_job& b) {
    const bool one_a = resident_tile_rows(a.rows, a.cols) != 0, one_b = resident_tile_rows(b.rows, b.cols) != 0;
    if (one_a && one_b) return false;
    return (!one_a || job_read(a) <= 16 << 20) && (!one_b || job_read(b) <= 16 << 20);
}
// tile_rows: 64 or 128, whole 128 x 128 tiles either way
static CastJob kernel_job(const f8mi_cast_job& j, int tile_rows) {
    CastJob k{};
    k.x = j.x; k.rows = j.rows; k.cols = j.cols; k.ld = j.ld; k.out = j.out; k.out_t = j.out_t;
    k.tiles_x = (uint32_t)((j.cols + CAST_TILE - 1) / CAST_TILE);
    k.tiles_y = (uint32_t)((j.rows + CAST_TILE - 1) / CAST_TILE) * (CAST_TILE / tile_rows);
    k.out_kb = j.out ? j.out_layout : F8MI_LAYOUT_ROWMAJOR;
    k.out_t_kb = j.out_t ? j.out_t_layout : F8MI_LAYOUT_ROWMAJOR;
    return k;
}
static double job_bytes(const f8mi_cast_job& j) {
    const double n = (double)j.rows * (double)j.cols;
    return (j.ld == 0 ? (double)j.cols : n) * (j.in_dtype == F8MI_FP32 ? 4 : 2) + n * ((j.out ? 1 : 0) + (j.out_t ? 1 : 0));
}

// tile_rows != 0: the resident kernel with such tiles; else the cast behind an amax launch, or, TAGGED, the delayed one
template <int DTA, int DTB, bool TAGGED>
static int launch_cast_pair1(int tile_rows, hipStream_t stream, const CastJob& a, const CastJob& b) {
    const uint32_t nb_a = a.tiles_x * a.tiles_y;
    const dim3 g(nb_a + b.tiles_x * b.tiles_y), t(CAST_THREADS);
    if constexpr (!TAGGED) {
        if (tile_rows == 64) hipLaunchKernelGGL((cast_dynamic_resident_pair_kernel<DTA, DTB, F8MI_E4M3FN, 1>), g, t, 0, stream, a, b, nb_a);
        else if (tile_rows == 128) hipLaunchKernelGGL((cast_dynamic_resident_pair_kernel<DTA, DTB, F8MI_E4M3FN, 2>), g, t, 0, stream, a, b, nb_a);
        // (unequal types: five workgroups a CU, and no fewer is faster)
        else hipLaunchKernelGGL((cast_pair_kernel<DTA, DTB, F8MI_E4M3FN, false>), g, t, DTA == DTB ? unused_lds(DTA, g.x) : 0u, stream, a, b, nb_a);
    } else {
        hipLaunchKernelGGL((cast_pair_kernel<DTA, DTB, F8MI_E4M3FN, true>), g, t, 0, stream, a, b, nb_a);
    }
    return check_hip(hipGetLastError(), "cast (two tensors) kernel launch");
}
template <bool TAGGED>
static int launch_cast_pair(int dt_a, int dt_b, int tile_rows, hipStream_t stream, const CastJob& a, const CastJob& b) {
    if (dt_a == F8MI_BF16 && dt_b == F8MI_BF16) return launch_cast_pair1<F8MI_BF16, F8MI_BF16, TAGGED>(tile_rows, stream, a, b);
    if (dt_a == F8MI_FP16 && dt_b == F8MI_FP16) return launch_cast_pair1<F8MI_FP16, F8MI_FP16, TAGGED>(tile_rows, stream, a, b);
    if (dt_a == F8MI_BF16 && dt_b == F8MI_FP32) return launch_cast_pair1<F8MI_BF16, F8MI_FP32, TAGGED>(tile_rows, stream, a, b);
    if (dt_a == F8MI_FP16 && dt_b == F8MI_FP32) return launch_cast_pair1<F8MI_FP16, F8MI_FP32, TAGGED>(tile_rows, stream, a, b);
    return launch_cast_pair1<F8MI_FP32, F8MI_FP32, TAGGED>(tile_rows, stream, a, b);
}


// Rows of the tiles that both get in one launch, 0: not in one.  Two 16-bit tensors may have half as many tiles again as one tensor (`large`): in two
// launches each of them waits for its own words, together once.  us, two launches / one: 2048 x 4096 with 3072 x 4096 (1280 tiles) 25.9 /
// 21.0, with 4096 x 4096 (1536) 29.1 / 24.1, both copies 33.1 / 26.7; 3000 x 3000 with 3100 x 3000, both copies 30.0 / 22.3; 1024 x 4096 with 5120 x 4096
// (two launches, one of them for the maxima) 26.0 / 24.3.  Six workgroups of eight leave other kernels a quarter of the chip.  Seven (1792 tiles) are
// faster alone and slower beside each other: 3072 x 4096 with 4096 x 4096 32.1 / 29.2, on two streams at once 27.2 / 31.8; 1024 x 4096 with
// 6144 x 4096 29.9 / 29.2 and 25.0 / 73.6.  fp32 has room for five.
static int pair_tile_rows(const f8mi_cast_job& a, const f8mi_cast_job& b, bool* large) {
    const int64_t tiles = tiles_of(a) + tiles_of(b);
    *large = false;
    if (const int rows = resident_tile_rows(tiles * CAST_TILE, CAST_TILE)) return rows;
    *large = b.in_dtype != F8MI_FP32 && tiles <= std::min(RESIDENT_PAIR_TILES, 6 * cu_count());
    return *large ? CAST_TILE : 0;
}
// Streams whose large pairs may be there at once.  us a pair of 2048 x 4096 with 4096 x 4096, two launches / one: on two streams 23.7 / 22.4, on
// three 23.4 / 45.8, both copies 28.4 / 56.1 (some hold the places that others wait for).
constexpr int LARGE_PAIR_STREAMS = 2;
// Both casts in the launch that exchanges maxima.  F8MI_ERR_UNSUPPORTED, and nothing queued: not in one.
static int cast_dynamic_pair_one_launch(const f8mi_cast_job& a, const f8mi_cast_job& b, uint32_t wait_ticks, hipStream_t stream, int large_pair_streams) {
    bool large;
    const int tile_rows = pair_tile_rows(a, b, &large);
    if (!tile_rows) return F8MI_ERR_UNSUPPORTED;
    TaggedWords tagged;
    int streams = 0;
    if (const int rc = begin_exchange(stream, wait_ticks, tagged, &streams)) return rc;
    if (!tagged.words || (large && streams > large_pair_streams)) return F8MI_ERR_UNSUPPORTED;
    CastJob ja = kernel_job(a, tile_rows), jb = kernel_job(b, tile_rows);
    ja.scale_out = a.scale_dev;
    jb.scale_out = b.scale_dev;
    ja.tagged = jb.tagged = tagged;
    jb.tagged.words += ja.tiles_x * ja.tiles_y;
    ProfScope prof(F8MI_K_CAST, job_bytes(a) + job_bytes(b), stream);
    return launch_cast_pair<false>(a.in_dtype, b.in_dtype, tile_rows, stream, ja, jb);
}
static int cast_delayed_pair_one_launch(const f8mi_cast_job& a, const f8mi_cast_job& b, uint32_t wait_ticks, hipStream_t stream) {
    if (!a.amax_dev || !b.amax_dev || !one_launch_delayed((tiles_of(a) + tiles_of(b)) * CAST_TILE, CAST_TILE)) return F8MI_ERR_UNSUPPORTED;
    TaggedWords tagged;
    if (const int rc = begin_exchange(stream, wait_ticks, tagged)) return rc;
    if (!tagged.words) return F8MI_ERR_UNSUPPORTED;
    CastJob ja = kernel_job(a, CAST_TILE), jb = kernel_job(b, CAST_TILE);
    ja.scale_dev = a.scale_dev;
    jb.scale_dev = b.scale_dev;
    ja.amax_out = a.amax_dev;
    jb.amax_out = b.amax_dev;
    ja.tagged = jb.tagged = tagged;
    jb.tagged.words += ja.tiles_x * ja.tiles_y * (CAST_THREADS / 64);
    ProfScope prof(F8MI_K_CAST, job_bytes(a) + job_bytes(b), stream);
    return launch_cast_pair<true>(a.in_dtype, b.in_dtype, 0, stream, ja, jb);
}

}  // namespace f8mi

extern "C" int f8mi_cast_one_launch(const f8mi_cast_job* a, const f8mi_cast_job* b, int delayed, uint32_t wait_ticks, void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (!a || !pair_ok(*a, b ? *b : *a) || (delayed && (!a->amax_dev || (b && !b->amax_dev)))) { set_error("f8mi_cast_one_launch: bad job"); return F8MI_ERR_INVALID_ARG; }
    int rc;
    if (b) rc = delayed ? cast_delayed_pair_one_launch(*a, *b, wait_ticks, stream) : cast_dynamic_pair_one_launch(*a, *b, wait_ticks, stream, EXCHANGE_STREAMS);
    else if (delayed) rc = cast_delayed_one_launch(a->x, a->rows, a->cols, a->ld, a->in_dtype, a->scale_dev, F8MI_E4M3FN, a->out, a->out_layout, a->out_t, a->out_t_layout, a->amax_dev, wait_ticks, stream);
    else return f8mi_cast_dynamic_resident(a->x, a->rows, a->cols, a->ld, a->in_dtype, F8MI_E4M3FN, a->scale_dev, a->out, a->out_layout, a->out_t, a->out_t_layout, wait_ticks, stream_);
    if (rc == F8MI_ERR_UNSUPPORTED) set_error("f8mi_cast_one_launch: more tiles than one launch takes, or a stream that is being captured");
    return rc;
}

extern "C" int f8mi_cast_dynamic_pair(const f8mi_cast_job* a, const f8mi_cast_job* b, void* workspace, void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (!a || !b) { set_error("f8mi_cast_dynamic_pair: null job"); return F8MI_ERR_INVALID_ARG; }
    if (workspace && (uintptr_t)workspace % 16 == 0 && pair_ok(*a, *b)) {
        const int one = cast_dynamic_pair_one_launch(*a, *b, EXCHANGE_WAIT_TICKS, stream, LARGE_PAIR_STREAMS);
        if (one != F8MI_ERR_UNSUPPORTED) return one;
        // one of them too large for a launch of its own: both through the two launches it takes
        if (two_launches_pay(*a, *b) && a->ld && b->ld &&
            amax_pair_ok(a->x, a->rows, a->cols, a->ld, b->x, b->rows, b->cols, b->ld)) {
            CastJob ja = kernel_job(*a, CAST_TILE), jb = kernel_job(*b, CAST_TILE);
            ja.scale_out = a->scale_dev;
            jb.scale_out = b->scale_dev;
            ja.amax_ws = (const uint32_t*)workspace;
            {
                ProfScope prof(F8MI_K_AMAX, (double)job_read(*a) + (double)job_read(*b), stream);
                if (const int rc = launch_amax_pair(a->in_dtype, b->in_dtype, a->x, a->rows * a->cols, b->x, b->rows * b->cols, (uint32_t*)workspace, stream, &jb.amax_ws,
                                                    &ja.amax_nblocks, &jb.amax_nblocks))
                    return rc;
            }
            ProfScope prof(F8MI_K_CAST, job_bytes(*a) + job_bytes(*b), stream);
            return launch_cast_pair<false>(a->in_dtype, b->in_dtype, 0, stream, ja, jb);
        }
    }
    for (const f8mi_cast_job* j : {a, b})
        if (const int rc = f8mi_cast_dynamic(j->x, j->rows, j->cols, j->ld, j->in_dtype, F8MI_E4M3FN, j->scale_dev, j->out, j->out_layout, j->out_t, j->out_t_layout, workspace, stream_))
            return rc;
    return F8MI_OK;
}

extern "C" int f8mi_cast_delayed_pair(const f8mi_cast_job* a, const f8mi_cast_job* b, void* workspace, void* stream_) {
    hipStream_t stream = (hipStream_t)stream_;
    if (!a || !b) { set_error("f8mi_cast_delayed_pair: null job"); return F8MI_ERR_INVALID_ARG; }
    if (pair_ok(*a, *b)) {
        const int rc = cast_delayed_pair_one_launch(*a, *b, EXCHANGE_WAIT_TICKS_LAST, stream);
        if (rc != F8MI_ERR_UNSUPPORTED) return rc;
    }
    for (const f8mi_cast_job* j : {a, b})
        if (const int rc = f8mi_cast_delayed(j->x, j->rows, j->cols, j->ld, j->in_dtype, j->scale_dev, F8MI_E4M3FN, j->out, j->out_layout, j->out_t, j->out_t_layout, j->amax_dev,
                                             workspace, stream_))
            return rc;
    return F8MI_OK;
}

namespace f8mi {

// ---- dynamic scaling for callers that cannot allocate ---------------------------------------------------------
// The per-workgroup partial maxima of the amax pass (one word per workgroup, at most WS_WORDS of them whatever the
// tensor's size) go to a device array that is part of the library's code object instead of a workspace the caller
// brings.  Every GPU holds its own copy of the array at its own address from the moment the library is loaded on
// it until the process ends; `scratch` below is only the host-side handle of it, the address is looked up once per
// device and kept.  Nothing in it has to start at zero: a call writes the words it reads back.
static __device__ __align__(256) uint32_t scratch[WS_WORDS];
static_assert(sizeof(scratch) == F8MI_STATIC_SCRATCH_BYTES, "f8mi.h states the size of the static scratch");

static std::atomic<uint32_t*> g_scratch_ptr[STATIC_MAX_DEVICES];

}  // namespace f8mi

extern "C" int f8mi_cast_dynamic_static(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, int fp8_fmt, float* scale_dev,
                                        uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout, void* stream) {
    if (rows < 0 || cols < 0) { set_error("f8mi_cast_dynamic_static: bad shape rows=%lld cols=%lld", (long long)rows, (long long)cols); return F8MI_ERR_INVALID_ARG; }
    if (rows > 0 && cols > F8MI_STATIC_MAX_ELEMS / rows) {
        set_error("f8mi_cast_dynamic_static: %lld x %lld elements, at most %lld per call (use f8mi_cast_dynamic with a workspace)",
                  (long long)rows, (long long)cols, (long long)F8MI_STATIC_MAX_ELEMS);
        return F8MI_ERR_INVALID_ARG;
    }
    uint32_t* ws = device_array(HIP_SYMBOL(scratch), g_scratch_ptr, "f8mi_cast_dynamic_static");
    if (!ws) return F8MI_ERR_HIP;
    return f8mi_cast_dynamic(x, rows, cols, ld, in_dtype, fp8_fmt, scale_dev, out, out_layout, out_t, out_t_layout, ws, stream);
}
