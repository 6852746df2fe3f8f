// Column sums of a tensor: the gradient of a bias.  HBM-bound: the tensor is read once, 16 bytes a lane, by enough workgroups to fill the
// chip whatever its shape: one takes 64 lanes' columns of one to several hundred rows (four waves, every fourth row each, eight loads in
// flight), writes fp32 partial sums, and a second launch adds those of a column in a fixed order.  us with both
// launches, torch's sum / this: 512 x 1024 9.0 / 6.3, 4096 x 4096 23.1 / 9.9 (fp32 24.5 / 15.2), 8192 x 1024 22.6 / 7.5, 4099 x 11007 (odd rows) 70 /
// 41, 16384 x 28672 172 / 141 (6.7 TB/s).
#include <algorithm>

#include "f8mi_gemm_util.h"

namespace f8mi {

constexpr int COLSUM_THREADS = 256, COLSUM_WAVES = COLSUM_THREADS / 64, COLSUM_UNROLL = 8;
constexpr int FINISH_WAVES = 16;
constexpr int COLSUM_MIN_ROWS = COLSUM_WAVES * COLSUM_UNROLL;  // of a workgroup: one batch of loads a wave

template <int DT>
struct ColsumCfg {
    static constexpr int V = DT == F8MI_FP32 ? 4 : 8;  // columns of a lane
    static constexpr int COLS = 64 * V;
};

template <int DT>
__device__ __forceinline__ void colsum_add(float (&s)[ColsumCfg<DT>::V], uint4 v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if constexpr (DT == F8MI_FP32) {
            s[i] += bits_to_float(w[i]);
        } else if constexpr (DT == F8MI_BF16) {
            s[2 * i] += bits_to_float(w[i] << 16);
            s[2 * i + 1] += bits_to_float(w[i] & 0xffff0000u);
        } else {
            s[2 * i] += fp16_bits_to_float((uint16_t)w[i]);
            s[2 * i + 1] += fp16_bits_to_float((uint16_t)(w[i] >> 16));
        }
    }
}

// The sum, rounded to x's type as torch's sum of such a tensor, in the type of the bias.
template <int DT>
__device__ __forceinline__ void colsum_store(float s, void* out, int out_dt, int64_t col) {
    if constexpr (DT == F8MI_BF16) s = bits_to_float(pack2<F8MI_BF16>(s, 0.f) << 16);
    if constexpr (DT == F8MI_FP16) s = fp16_bits_to_float((uint16_t)pack2<F8MI_FP16>(s, 0.f));
    if (out_dt == F8MI_FP32) ((float*)out)[col] = s;
    else if (out_dt == F8MI_BF16) ((uint16_t*)out)[col] = (uint16_t)pack2<F8MI_BF16>(s, 0.f);
    else ((uint16_t*)out)[col] = (uint16_t)pack2<F8MI_FP16>(s, 0.f);
}

template <int DT>
__global__ __launch_bounds__(COLSUM_THREADS) void colsum_kernel(const uint8_t* __restrict__ x, int64_t rows, int64_t cols, int64_t ld, int64_t chunk_rows,
                                                                float* __restrict__ partial, void* __restrict__ out, int out_dt) {
    constexpr int V = ColsumCfg<DT>::V, COLS = ColsumCfg<DT>::COLS, SIZE = DT == F8MI_FP32 ? 4 : 2;
    __shared__ float red[COLSUM_WAVES][COLS];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t col = (int64_t)blockIdx.x * COLS + lane * V;
    const int64_t first = blockIdx.y * chunk_rows, end = min(first + chunk_rows, rows);
    float s[V];
#pragma unroll
    for (int i = 0; i < V; i++) s[i] = 0.f;
    int64_t r = first + wave;
    if (col + V <= cols) {
        const uint8_t* p = x + (r * ld + col) * SIZE;
        const int64_t step = COLSUM_WAVES * ld * SIZE;
        for (; r + (COLSUM_UNROLL - 1) * COLSUM_WAVES < end; r += COLSUM_UNROLL * COLSUM_WAVES) {
            uint4 v[COLSUM_UNROLL];
#pragma unroll
            for (int u = 0; u < COLSUM_UNROLL; u++, p += step) v[u] = load_nt16_any(p);
#pragma unroll
            for (int u = 0; u < COLSUM_UNROLL; u++) colsum_add<DT>(s, v[u]);
        }
        for (; r < end; r += COLSUM_WAVES, p += step) colsum_add<DT>(s, load_nt16_any(p));
    } else if (col < cols) {  // the last lane with columns may have fewer than its eight or four
        for (; r < end; r += COLSUM_WAVES)
#pragma unroll
            for (int i = 0; i < V; i++)
                if (col + i < cols) s[i] += load_bias<DT>(x + r * ld * SIZE, (int)(col + i));
    }
#pragma unroll
    for (int i = 0; i < V; i++) red[wave][lane * V + i] = s[i];
    __syncthreads();
#pragma unroll
    for (int i = threadIdx.x; i < COLS; i += COLSUM_THREADS) {
        const int64_t c = (int64_t)blockIdx.x * COLS + i;
        if (c >= cols) break;
        const float sum = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
        if (partial) partial[blockIdx.y * cols + c] = sum;
        else colsum_store<DT>(sum, out, out_dt, c);
    }
}

// 64 columns a workgroup, a wave every 16th of their partial sums (four waves: 16384 x 512 12.1 us)
template <int DT>
__global__ __launch_bounds__(64 * FINISH_WAVES) void colsum_finish_kernel(const float* __restrict__ partial, int64_t chunks, int64_t cols, void* __restrict__ out,
                                                                       int out_dt) {
    __shared__ float red[FINISH_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t col = (int64_t)blockIdx.x * 64 + lane;
    float s = 0.f;
    if (col < cols) {
#pragma unroll 8
        for (int64_t i = wave; i < chunks; i += FINISH_WAVES) s += partial[i * cols + col];
    }
    red[wave][lane] = s;
    __syncthreads();
    if (wave != 0 || col >= cols) return;
    s = red[0][lane];
#pragma unroll
    for (int i = 1; i < FINISH_WAVES; i++) s += red[i][lane];
    colsum_store<DT>(s, out, out_dt, col);
}

// Rows of a workgroup: 1024 workgroups, four on a CU, unless there are too few rows (us with 512 / 1024 / 2048: 4096 x 4096 11.4 / 10.6 / 10.6, fp32
// 20.2 / 14.7 / 15.5, 4099 x 11007 55 / 41 / 35, 8192 x 14336 38.8 / 40.6 / 40.0).
static int64_t colsum_chunk_rows(int64_t rows, int64_t cols, int dtype) {
    const int64_t width = dtype == F8MI_FP32 ? ColsumCfg<F8MI_FP32>::COLS : ColsumCfg<F8MI_BF16>::COLS;
    const int64_t strips = (cols + width - 1) / width, want = std::max<int64_t>(1, 1024 / strips);
    const int64_t each = (rows + want - 1) / want;
    return std::max<int64_t>(1, (each + COLSUM_MIN_ROWS - 1) / COLSUM_MIN_ROWS) * COLSUM_MIN_ROWS;
}

template <int DT>
static int launch_colsum(const void* x, int64_t rows, int64_t cols, int64_t ld, void* out, int out_dtype, float* ws, hipStream_t stream) {
    const int64_t chunk_rows = colsum_chunk_rows(rows, cols, DT), chunks = (rows + chunk_rows - 1) / chunk_rows;
    const unsigned strips = (unsigned)((cols + ColsumCfg<DT>::COLS - 1) / ColsumCfg<DT>::COLS);
    hipLaunchKernelGGL(colsum_kernel<DT>, dim3(strips, (unsigned)chunks), dim3(COLSUM_THREADS), 0, stream, (const uint8_t*)x, rows, cols, ld, chunk_rows,
                       chunks > 1 ? ws : nullptr, out, out_dtype);
    if (chunks > 1)
        hipLaunchKernelGGL(colsum_finish_kernel<DT>, dim3((unsigned)((cols + 63) / 64)), dim3(64 * FINISH_WAVES), 0, stream, ws, chunks, cols, out, out_dtype);
    return check_hip(hipGetLastError(), "column sum kernel launch");
}

}  // namespace f8mi

using namespace f8mi;

extern "C" int64_t f8mi_column_sum_workspace_bytes(int64_t rows, int64_t cols, int dtype) {
    if (rows <= 0 || cols <= 0) return 0;
    const int64_t chunk_rows = colsum_chunk_rows(rows, cols, dtype), chunks = (rows + chunk_rows - 1) / chunk_rows;
    return chunks > 1 ? chunks * cols * 4 : 0;
}

extern "C" int f8mi_column_sum(const void* x, int64_t rows, int64_t cols, int64_t ld, int dtype, void* out, int out_dtype, void* workspace,
                               int64_t workspace_bytes, void* stream) {
    if (rows <= 0 || cols <= 0 || ld < cols || cols > 0x7fffffff) { set_error("f8mi_column_sum: bad shape rows=%lld cols=%lld ld=%lld", (long long)rows, (long long)cols, (long long)ld); return F8MI_ERR_INVALID_ARG; }
    if (dtype < 0 || dtype > 2 || out_dtype < 0 || out_dtype > 2) { set_error("f8mi_column_sum: unknown dtype code"); return F8MI_ERR_INVALID_ARG; }
    const int64_t need = f8mi_column_sum_workspace_bytes(rows, cols, dtype);
    if (!x || !out || (need && (!workspace || workspace_bytes < need || (uintptr_t)workspace % 4 != 0))) { set_error("f8mi_column_sum: null pointer or a workspace that is too small"); return F8MI_ERR_INVALID_ARG; }
    if (dtype == F8MI_BF16) return launch_colsum<F8MI_BF16>(x, rows, cols, ld, out, out_dtype, (float*)workspace, (hipStream_t)stream);
    if (dtype == F8MI_FP16) return launch_colsum<F8MI_FP16>(x, rows, cols, ld, out, out_dtype, (float*)workspace, (hipStream_t)stream);
    return launch_colsum<F8MI_FP32>(x, rows, cols, ld, out, out_dtype, (float*)workspace, (hipStream_t)stream);
}
