/*
 * f8mi.h -- C ABI of libf8mi.so: the Float8Linear training hot path of
 * pytorch-labs/float8_experimental as hand-written gfx950 (MI355X) kernels.
 *
 * Conventions
 *   - Every pointer named `*_dev`, every tensor pointer and every workspace is
 *     DEVICE memory owned by the caller.  The library never allocates, frees or
 *     synchronises; every call only enqueues kernels on `stream` (a
 *     hipStream_t passed as void*; NULL = the default stream).
 *   - Calls are re-entrant and may come from any host thread (autograd runs the
 *     backward on its own thread).
 *   - Return value: F8MI_OK or a negative F8MI_ERR_* code; f8mi_last_error()
 *     gives the calling thread's last message.
 *   - "scale" always has the reference's meaning: high precision * scale = fp8
 *     range (float8_tensor.py:252-255 of the reference).
 *
 * Paths cited below are relative to the reference checkout
 * (pytorch-labs/float8_experimental).
 */
#ifndef F8MI_H
#define F8MI_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define F8MI_VERSION 130

#define F8MI_OK 0
#define F8MI_ERR_INVALID_ARG (-1) /* null pointer, negative size, unknown enum            */
#define F8MI_ERR_UNSUPPORTED (-2) /* valid request this build does not implement          */
#define F8MI_ERR_HIP (-3)         /* a HIP runtime call failed (launch, event, ...)       */
#define F8MI_ERR_ARCH (-4)        /* the current device is not gfx950                     */

/* element type of a high-precision tensor, and the dtype arithmetic is rounded to */
#define F8MI_BF16 0
#define F8MI_FP16 1
#define F8MI_FP32 2

/* OCP fp8 formats (torch.float8_e4m3fn / torch.float8_e5m2; float8_utils.py:31-32) */
#define F8MI_E4M3FN 0
#define F8MI_E5M2 1

/* kernel ids for the profiling counters */
#define F8MI_K_AMAX 0
#define F8MI_K_CAST 1
#define F8MI_K_GEMM 2
#define F8MI_K_SYNC 3
#define F8MI_K_COUNT 4

int f8mi_version(void);
const char* f8mi_last_error(void);

/* "" for the library as shipped.  A measurement build (compiled with one of the knobs of csrc/f8mi_knobs.h set: another
 * tile walk, cache policy, ...) answers with the knobs' names and values, so that callers and benchmarks can tell
 * and record which build they run.  Every knob leaves results unchanged.  No counterpart in the reference. */
const char* f8mi_build_knobs(void);

/* Fills CU count, LDS bytes per workgroup and the gcn arch name of HIP device `device`.
 * Returns F8MI_ERR_ARCH when it is not a gfx950. */
int f8mi_device_info(int device, int* cu_count, int* lds_bytes, char* arch, int arch_len);

/* Bytes of the small device workspace f8mi_amax_scale needs (per-block partial
 * results; 4 KB).  Its contents between calls do not matter.  One workspace must
 * not be shared by calls that can overlap in time (use one per stream). */
size_t f8mi_workspace_bytes(void);

/*
 * amax = max|x| and the fp8 scale derived from it, in one pass over x.
 * Replaces tensor_to_amax (float8_utils.py:102-112) + amax_to_scale
 * (float8_utils.py:35-57), i.e. tensor_to_scale (float8_utils.py:115-120).
 *   x          rows x cols elements of `in_dtype`, row stride `ld` elements (ld >= cols), or ld = 0: every row is
 *              the same `cols` elements -- a broadcast row, as autograd hands an expanded gradient
 *              (float8_scaling_utils.py:204-216 receives y.sum().backward()'s dY that way); f8mi_cast and
 *              f8mi_cast_dynamic take ld = 0 likewise, and only `cols` elements are read
 *   math_dtype dtype each step of `fmax / clamp(amax, 1e-12)` is rounded to:
 *              `in_dtype` for dynamic scaling (the reference computes the scale
 *              in the tensor's dtype), F8MI_FP32 for delayed-scaling buffers
 *   orig_is_fp16  clamp the scale to 65504 (float8_utils.py:54-55)
 *   amax_dev   out, 1 float (the amax widened to fp32), may be NULL
 *   scale_dev  out, 1 float, may be NULL
 * NaN anywhere in x gives NaN amax and NaN scale, like torch.max.
 */
int f8mi_amax_scale(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, int fp8_fmt,
                    int math_dtype, int orig_is_fp16, float* amax_dev, float* scale_dev, void* workspace,
                    void* stream);

/* One tensor of a list given to f8mi_amax_scale_multi. */
typedef struct f8mi_tensor_ref {
    const void* data;   /* dense, 16-byte aligned, `numel` elements of the call's in_dtype */
    int64_t numel;
    int64_t first_tile; /* number of tiles of all entries before this one; an entry has
                           numel / f8mi_amax_tile_elems(in_dtype) + 1 tiles */
} f8mi_tensor_ref;

/* Elements of `in_dtype` in one tile (32 KB) of f8mi_amax_scale_multi's numbering. */
int64_t f8mi_amax_tile_elems(int in_dtype);

/*
 * amax and scale of n tensors in one pass: amax_dev[i], scale_dev[i] (either may be NULL) as
 * f8mi_amax_scale gives them for tensor i.  Replaces the torch._foreach_norm(weights, ord=inf)
 * + stack + clamp + divide chain of precompute_float8_dynamic_scale_for_fsdp
 * (fsdp_utils.py:59-66) -- the per-GPU part of it; the all-reduce between ranks is the caller's.
 *   refs_dev     device array of n entries (n <= f8mi_workspace_bytes() / 4)
 *   total_tiles  sum of the entries' tile counts
 * Three launches whatever n is.
 */
int f8mi_amax_scale_multi(const f8mi_tensor_ref* refs_dev, int n, int64_t total_tiles, int in_dtype, int fp8_fmt,
                          int math_dtype, int orig_is_fp16, float* amax_dev, float* scale_dev, void* workspace,
                          void* stream);

/*
 * Saturated cast to fp8: bytes = fp8(clamp(x * scale, -fmax, fmax)), round to
 * nearest even.  Replaces _ToFloat8ConstrFunc.forward (float8_tensor.py:139-191)
 * + to_fp8_saturated (float8_utils.py:123-139), and the fp8 transpose copies
 * that preprocess_addmm makes for the backward GEMMs (float8_ops.py:131-155).
 *   scale_dev      1 float in device memory
 *   product_dtype  dtype `x * scale` is rounded to before clamp + conversion:
 *                  `in_dtype` when the reference's scale is a 0-dim tensor
 *                  (dynamic scaling), F8MI_FP32 when it is the [1]-shaped buffer
 *                  of delayed scaling or x is fp32
 *   out            rows x cols bytes, dense row-major; may be NULL
 *   out_t          cols x rows bytes, dense (the transpose); may be NULL
 *   amax_dev       if not NULL, max|x| of THIS call is stored there (fused
 *                  amax for hp_tensor_to_float8_delayed,
 *                  float8_scaling_utils.py:65-96)
 *   workspace      reserved; may be NULL
 */
int f8mi_cast(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, const float* scale_dev,
              int product_dtype, int fp8_fmt, uint8_t* out, uint8_t* out_t, float* amax_dev, void* workspace,
              void* stream);

/*
 * C[m][n] = (sum_k A[m][k] * Bt[n][k]) * (1/scale_a) * (1/scale_b) (+ bias[n]),
 * fp32 accumulation on the fp8 matrix cores.  Replaces addmm_float8_unwrapped
 * -> torch._scaled_mm (float8_python_api.py:24-64) as reached from float8_mm
 * (float8_ops.py:158-190).  Both operands are contiguous along k (A row-major,
 * B column-major in the reference's words): forward x*W^T, grad_input dY*W and
 * grad_weight dY^T*x all have this form once the transposed copies exist.
 * Any m, n, k >= 0 is accepted (ragged edges are handled in the kernel).  Up to 16 rows of A (up to 256
 * while streaming Bt once per 128 rows beats a round of 128-row tiles: a narrow Bt) with k % 128 == 0 take a
 * kernel that reads Bt at memory speed (an inference decode step); it sums the products in another order
 * than the tile kernels, so its results agree with theirs within the accumulation tolerance, not bit for bit.
 * Which kernel runs depends on (m, n, k) and alignment only.
 *   a_fmt/b_fmt   F8MI_E4M3FN / F8MI_E5M2 per operand
 *   lda/ldb       row strides in bytes (>= k)
 *   scale_a_dev, scale_b_dev   the operands' forward scales (1 float each)
 *   c_dtype       F8MI_BF16 / F8MI_FP16 / F8MI_FP32, ldc in elements
 *   bias_dev      n elements of c_dtype, or NULL
 */
int f8mi_gemm_nt(const void* a, int a_fmt, int64_t lda, const void* bt, int b_fmt, int64_t ldb, int64_t m,
                 int64_t n, int64_t k, const float* scale_a_dev, const float* scale_b_dev, void* c, int c_dtype,
                 int64_t ldc, const void* bias_dev, void* stream);

/* ---- k-blocked operands: the layout the fused Float8Linear path keeps its fp8 copies in ----
 * A GEMM operand with R rows and contraction length kc (a multiple of 64) is stored as
 * [kc/64][R][64]: byte (r, k) sits at ((k/64)*R + r)*64 + k%64.  The 64-deep slab of 256 rows
 * that a workgroup consumes per step is then 16 KB of consecutive memory instead of 256 pieces
 * of 64 bytes, which the load unit and the L2 move measurably faster (whole cache lines, even
 * channel spread).  The reference keeps fp8 data row-major only (float8_tensor.py:250-262,
 * float8_ops.py:150-153); these two entry points have no counterpart there and never change
 * values, only where bytes are put.
 */
#define F8MI_LAYOUT_ROWMAJOR 0
#define F8MI_LAYOUT_KBLOCK64 1
/* The same layout for ANY contraction length: the contraction is extended with zero bytes to f8mi_padded_k(kc), the
 * next multiple of 128, and stored [f8mi_padded_k(kc)/64][R][64].  Zeros add nothing to a product, so a GEMM over the
 * padded length gives the product of the unpadded operands -- what the reference's pad_tensor_for_matmul does to the
 * inner dimension of a ragged layer before torch._scaled_mm (float8_utils.py:206-247, float8_ops.py:139-149), here
 * done by the cast kernel as it writes the copy.  Output only: the GEMM entry points take such an operand as an
 * ordinary k-blocked one of contraction length f8mi_padded_k(kc). */
#define F8MI_LAYOUT_KBLOCK64_PAD128 2

/* Contraction length of a F8MI_LAYOUT_KBLOCK64_PAD128 operand: k rounded up to a multiple of 128 (pure arithmetic). */
int64_t f8mi_padded_k(int64_t k);

/* f8mi_cast with a layout per output.  out_layout = KBLOCK64 stores `out` as [cols/64][rows][64]
 * (needs cols % 64 == 0), out_t_layout = KBLOCK64 stores the transpose as [rows/64][cols][64]
 * (needs rows % 64 == 0).  KBLOCK64_PAD128 takes any shape: `out` is [f8mi_padded_k(cols)/64][rows][64] and `out_t`
 * [f8mi_padded_k(rows)/64][cols][64] bytes, every byte of which is written (zeros past the tensor's edge, also
 * when the scale is NaN).  The input's rows need no alignment beyond the element's own: eight elements are one
 * 16-byte load at any row pitch.  Everything else as f8mi_cast. */
int f8mi_cast_layout(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, const float* scale_dev,
                     int product_dtype, int fp8_fmt, uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout,
                     float* amax_dev, void* stream);

/* Delayed scaling in one call: f8mi_cast_layout with the module's existing scale (the product x * scale in fp32, as
 * with the [1]-shaped scale buffer), and *amax_dev = max|x| of this call -- hp_tensor_to_float8_delayed
 * (float8_scaling_utils.py:65-96: amax_buffer.fill_(tensor_to_amax(x)), then the cast with the stale scale).
 * Same bytes and the same amax as f8mi_cast_layout with amax_dev; what differs is how the amax leaves the cast kernel:
 * there every workgroup compares with *amax_dev at its end (and holds its LDS and wave slots for that round trip:
 * 6 - 20 us per tensor of 128 MB - 1.8 GB).  Here, up to 2048 tiles of 128 x 128 and unless the stream is being captured, every wave
 * leaves its maximum in a word of the library's own, and the workgroup started last collects them; beyond, every wave
 * folds it into one of 1024 words of `workspace` with an atomic that returns nothing, and a one-workgroup launch reduces
 * the words (4 us).
 *   workspace   f8mi_delayed_workspace_bytes() of device memory, 4-byte aligned, ALL ZERO before the first call that
 *               uses it; every call leaves it all zero again when its work completes.  Not to be shared by calls that
 *               can overlap in time (one per stream), and not the workspace of f8mi_amax_scale, whose contents are
 *               arbitrary. */
size_t f8mi_delayed_workspace_bytes(void);
int f8mi_cast_delayed(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, const float* scale_dev, int fp8_fmt,
                      uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout, float* amax_dev, void* workspace,
                      void* stream);

/* Dynamic scaling in one call: scale = f8mi_amax_scale(x) in x's own dtype, then f8mi_cast_layout(x, scale) with the
 * product in x's dtype -- hp_tensor_to_float8_dynamic (float8_scaling_utils.py:33-62: tensor_to_scale, then
 * hp_tensor_and_scale_to_float8 with the 0-dim scale).  *scale_dev receives the scale.  A tensor of at most
 * 32 K elements goes through one launch of one workgroup (a few rows of activations: the launches cost more
 * than the work), a dense one of at most 320 KB (of few rows: 512 KB) of which one copy is asked for through one launch of
 * several, anything else of at most 1024 tiles of 128 x 128 through f8mi_cast_dynamic_resident unless the stream is being
 * captured, and the rest through the two kernels above; the results are the same bits either way.
 * `workspace` as for f8mi_amax_scale. */
int f8mi_cast_dynamic(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, int fp8_fmt, float* scale_dev,
                      uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout, void* workspace, void* stream);

/* f8mi_cast_dynamic without the workspace argument, for callers that cannot allocate device memory (code under HIP
 * graph capture, tight serving loops, harnesses that forbid hipMalloc) and so have no workspace to bring.  No
 * counterpart in the reference.  The per-workgroup partial maxima go to an array of F8MI_STATIC_SCRATCH_BYTES that is
 * part of the library's device code: every GPU the library runs on holds it from load until the process ends.  The
 * call allocates and frees nothing (the first call on a device looks the array's address up, once).  Same kernels,
 * same result bits as f8mi_cast_dynamic.  All calls on one GPU share the one array: calls that can overlap in time
 * on the same GPU (two streams, two host threads) race on it -- give such callers f8mi_cast_dynamic and a workspace
 * each.  The array keeps the last call's contents; nothing in it needs to start at zero.  Tensors of more than
 * F8MI_STATIC_MAX_ELEMS elements are refused with F8MI_ERR_INVALID_ARG.
 * The first call on a device asks the runtime for the array's address on the device that is current (which, as for
 * every entry point, must be the device `stream` belongs to); that query may load the library's code onto the device
 * and is not something to do while a stream is being captured.  Make one ordinary call on each device before the
 * first capture (any size will do); from then on the entry point only launches kernels and may be captured and
 * replayed. */
#define F8MI_STATIC_SCRATCH_BYTES 4096
#define F8MI_STATIC_MAX_ELEMS (1ll << 36)
int f8mi_cast_dynamic_static(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, int fp8_fmt,
                             float* scale_dev, uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout,
                             void* stream);

/* f8mi_cast_dynamic in one launch that reads x once, for tensors that the chip holds: at most 1024 tiles of 128 x 128 (fewer
 * on a device of fewer than 256 CUs).  f8mi_cast_dynamic takes it by itself; the same bits.  The workgroups exchange their
 * maxima inside the launch; one that has waited wait_ticks of the 100 MHz clock for the others reads the tiles itself whose
 * maxima are missing, so the launch ends and is right whatever else runs (wait_ticks 0: nobody waits).  Refused with
 * F8MI_ERR_UNSUPPORTED, nothing queued: larger tensors, a stream that is being captured. */
int f8mi_cast_dynamic_resident(const void* x, int64_t rows, int64_t cols, int64_t ld, int in_dtype, int fp8_fmt,
                               float* scale_dev, uint8_t* out, int out_layout, uint8_t* out_t, int out_t_layout,
                               uint32_t wait_ticks, void* stream);

/* One tensor of a call that casts two: the arguments of f8mi_cast_dynamic (scale_dev: written; amax_dev unused) or of
 * f8mi_cast_delayed (scale_dev: read). */
typedef struct f8mi_cast_job {
    const void* x;
    int64_t rows, cols, ld;
    float* scale_dev;
    uint8_t* out;
    uint8_t* out_t;
    float* amax_dev;
    int in_dtype, out_layout, out_t_layout;
} f8mi_cast_job;

/* f8mi_cast_dynamic of `a`, then of `b`, both to e4m3: the same bits, in one launch where the chip holds both (at most 1024 tiles
 * together, 1536 of 16-bit types while at most two streams make such casts), in two instead of three or four where one is larger than that.  Everything else is the two calls. */
int f8mi_cast_dynamic_pair(const f8mi_cast_job* a, const f8mi_cast_job* b, void* workspace, void* stream);
/* f8mi_cast_delayed of `a`, then of `b`, both to e4m3, in one launch up to 2048 tiles together. */
int f8mi_cast_delayed_pair(const f8mi_cast_job* a, const f8mi_cast_job* b, void* workspace, void* stream);
/* The one launch of these two, or, with b null, of f8mi_cast_dynamic_resident and of f8mi_cast_delayed (to e4m3), by itself, with wait_ticks as
 * there (in a delayed cast one workgroup collects, and reads the whole tensor when it gives up).  F8MI_ERR_UNSUPPORTED, nothing
 * queued, where they do not take it. */
int f8mi_cast_one_launch(const f8mi_cast_job* a, const f8mi_cast_job* b, int delayed, uint32_t wait_ticks, void* stream);

/* A whole linear of at most 16 rows and F8MI_FEW_ROWS_ELEMS activations in one kernel: c[m][n] = sum_k x8[m][k] * w[n][k]
 * / (scale_x * scale_w) (+ bias[n]) with x8 the saturated e4m3 cast of x, which every workgroup makes for itself.  The same
 * bits as f8mi_cast_dynamic (scale_x_dev null) or f8mi_cast_layout (scale_x_dev given, product in product_dtype) followed by
 * f8mi_gemm_nt / f8mi_gemm_nt_kb.  x: rows of ldx elements at element alignment; w: row-major (w_layout
 * F8MI_LAYOUT_ROWMAJOR, rows of k bytes) or k-blocked (F8MI_LAYOUT_KBLOCK64), 16-byte aligned; c in x's dtype.
 * F8MI_ERR_UNSUPPORTED, with nothing queued: more rows or activations, k % 128 != 0, an unaligned weight; fp32
 * with a k-blocked weight of more than 2^26 - 256 rows. */
#define F8MI_FEW_ROWS_ELEMS 32768
int f8mi_linear_few_rows(const void* x, int64_t ldx, int dtype, const float* scale_x_dev, int product_dtype, const void* w,
                         int w_fmt, int w_layout, const float* scale_w_dev, int64_t m, int64_t n, int64_t k, void* c,
                         int64_t ldc, const void* bias_dev, void* stream);

/* Weight-only inference for few rows: c[m][n] = sum_k x[m][k] * W[n][k] with x, c and W = w / *scale_dev in `dtype`,
 * the fp8 weight w (rows of ldw bytes) dequantised in registers: the quotient is taken in fp32 and rounded to `dtype`,
 * as torch divides (the scale rounded to `dtype` before); fp32 accumulation.  Any k >= 1, any alignment of rows to the
 * element size.  Replaces to_original_precision + linear (reference inference.py:104-107). */
int f8mi_gemm_weight_only(const void* x, int64_t ldx, int dtype, const uint8_t* w, int fp8_fmt, int64_t ldw, int64_t m,
                          int64_t n, int64_t k, const float* scale_dev, void* c, int64_t ldc, void* stream);
/* out[i] = in[i] / *scale_dev in `dtype`, the same quotient, for n consecutive elements (float8_tensor.py:198-212 of the
 * reference). */
int f8mi_dequant(const uint8_t* in, int fp8_fmt, int64_t n, const float* scale_dev, int dtype, void* out, void* stream);

/* f8mi_gemm_nt on k-blocked operands: a = [k/64][m][64], bt = [k/64][n][64], both 16-byte
 * aligned.  Needs k % 64 == 0 and k >= 384 (F8MI_ERR_UNSUPPORTED otherwise: keep such operands
 * row-major and call f8mi_gemm_nt).  Same arithmetic, same result bits as f8mi_gemm_nt. */
int f8mi_gemm_nt_kb(const void* a, int a_fmt, const void* bt, int b_fmt, int64_t m, int64_t n, int64_t k,
                    const float* scale_a_dev, const float* scale_b_dev, void* c, int c_dtype, int64_t ldc,
                    const void* bias_dev, void* stream);

/* f8mi_gemm_nt / f8mi_gemm_nt_kb with scratch memory for the library to use: `workspace` (16-byte aligned device
 * memory, `workspace_bytes` long, contents irrelevant before and after; calls sharing it must not overlap) lets an
 * output of few tiles with a long k be computed with k split over workgroups -- an inference linear with 17 to a few
 * hundred rows and a long contraction, which would otherwise leave most CUs idle: partial sums go to the workspace
 * and a second kernel adds them in a fixed order (deterministic; another summation order than without the split,
 * so the two agree within the accumulation tolerance, not bit for bit).  Which path runs depends on (m, n, k),
 * alignment (of the operands and of C's rows) and workspace_bytes only; F8MI_GEMM_WORKSPACE_BYTES is enough for every case that is ever split.
 * With workspace NULL they are f8mi_gemm_nt / f8mi_gemm_nt_kb.  No counterpart in the reference (torch._scaled_mm
 * hides hipBLASLt's own workspace, float8_python_api.py:24-64). */
#define F8MI_GEMM_WORKSPACE_BYTES (32ll << 20)
int f8mi_gemm_nt_ws(const void* a, int a_fmt, int64_t lda, const void* bt, int b_fmt, int64_t ldb, int64_t m,
                    int64_t n, int64_t k, const float* scale_a_dev, const float* scale_b_dev, void* c, int c_dtype,
                    int64_t ldc, const void* bias_dev, void* workspace, int64_t workspace_bytes, void* stream);
int f8mi_gemm_nt_kb_ws(const void* a, int a_fmt, const void* bt, int b_fmt, int64_t m, int64_t n, int64_t k,
                       const float* scale_a_dev, const float* scale_b_dev, void* c, int c_dtype, int64_t ldc,
                       const void* bias_dev, void* workspace, int64_t workspace_bytes, void* stream);

/* Which kernel f8mi_gemm_nt(_ws) / f8mi_gemm_nt_kb(_ws) would run for an m x n x k product (no GPU needed; for tests,
 * logs and benchmarks) into a dense 16-bit C.  (Where n is odd, an fp32 C, or one whose rows all start at multiples of four
 * bytes, may take F8MI_PLAN_TILES256X224 instead of 256 x 256 tiles: the same bits.)  `aligned`: operands and row strides are 16-byte aligned (k-blocked operands always are);
 * workspace_bytes: 0 without a workspace.  Returns a F8MI_PLAN_* code in bits 0-7, the number of parts k is split
 * into in bits 8-15 and, where 128-row tiles take part, 1 (128 x 128) or 2 (128 x 256) in bits 16-23; 0 for an
 * empty product.  No counterpart in the reference. */
#define F8MI_PLAN_TILES128_SPLIT_K 1 /* 128-row tiles, k split over workgroups, second kernel adds the parts */
#define F8MI_PLAN_FEW_ROWS 2         /* Bt streamed once per 128 rows, k split over the waves of a workgroup */
#define F8MI_PLAN_TILES128 3         /* 128 x 128 or 128 x 256 tiles */
#define F8MI_PLAN_TILES256 4         /* 256 x 256 tiles, 16x16x128 MFMA, operands through LDS-DMA */
#define F8MI_PLAN_TILES256_AND_128 5 /* the same for the tile rows of whole rounds, 128-row tiles for the rest */
#define F8MI_PLAN_TILES256_MFMA32 6  /* 256 x 256 tiles, 32x32x64 MFMA (k % 128 == 64) */
#define F8MI_PLAN_TILES256X224 8     /* 256 x 224 tiles, 16x16x128 MFMA, where they fill whole rounds better */
#define F8MI_PLAN_STAGED 7           /* 256 x 256 tiles, register-staged (ragged or short k, unaligned operands) */
int f8mi_gemm_plan(int64_t m, int64_t n, int64_t k, int aligned, int64_t workspace_bytes);

/* f8mi_gemm_nt_kb with operands that may be given transposed, so that one k-blocked copy of a tensor serves
 * both GEMMs that use it (no transposed fp8 copies at all):
 *   a, a_transposed = 0: [k/64][m][64] as above;  = 1: [m/64][k][64], i.e. the matrix [k][m] k-blocked over m
 *   bt likewise with n.
 * Forward x*W^T takes (0, 0); grad_input dY*W takes a = dY8 [n_out/64][tokens][64] (0) and bt = the forward's
 * W8 [k_in/64][n_out][64] (1); grad_weight dY^T*x takes a = that dY8 (1) and bt = the forward's x8 (1).
 * (1, 0) is not built.  Transposed operands need k % 128 == 0, k >= 384 and the operand's row count (m or n)
 * to be a multiple of 64.  Same result bits as f8mi_gemm_nt on the row-major operands (for m > 256: the
 * few-row kernel of f8mi_gemm_nt is not used for transposed operands). */
int f8mi_gemm_kb_ex(const void* a, int a_fmt, int a_transposed, const void* bt, int b_fmt, int b_transposed, int64_t m,
                    int64_t n, int64_t k, const float* scale_a_dev, const float* scale_b_dev, void* c, int c_dtype,
                    int64_t ldc, const void* bias_dev, void* stream);

/* f8mi_gemm_nt_kb of two e4m3 operands with the bias added to the finished product: rounded to C's type, the bias (of that type, or fp32
 * and rounded to it) added, the sum rounded again, the bits of the product followed by a pass that adds the bias.  k % 128 == 0 and the
 * products that f8mi_gemm_plan gives to 128-row, 256 x 256 or 256 x 224 tiles, workspace_bytes as there; F8MI_ERR_UNSUPPORTED, nothing
 * queued, for all others. */
int f8mi_gemm_kb_bias(const void* a, const void* bt, int64_t m, int64_t n, int64_t k, const float* scale_a_dev, const float* scale_b_dev,
                      void* c, int c_dtype, int64_t ldc, const void* bias_dev, int bias_dtype, int64_t workspace_bytes, void* stream);

/* out[j] = the sum of column j of x [rows][cols] (rows `ld` elements apart, unit column stride): fp32 sums in a fixed order, rounded to
 * x's type and stored in out_dtype: the gradient of a bias.  workspace: f8mi_column_sum_workspace_bytes (0: none needed). */
int f8mi_column_sum(const void* x, int64_t rows, int64_t cols, int64_t ld, int dtype, void* out, int out_dtype, void* workspace,
                    int64_t workspace_bytes, void* stream);
int64_t f8mi_column_sum_workspace_bytes(int64_t rows, int64_t cols, int dtype);

/* Types of C beside those of tensors, for the second product of f8mi_gemm_pair beside a first one of the 16-bit type: fp32 that holds the product rounded to the 16-bit type, the bits of such a product
 * followed by a conversion (the gradient of an fp32 weight under autocast). */
#define F8MI_BF16_IN_FP32 3
#define F8MI_FP16_IN_FP32 4

/* One product of a call that computes two: the arguments of f8mi_gemm_kb_ex without a bias and, for operands that are both given as they
 * are, the workspace of f8mi_gemm_nt_kb_ws. */
typedef struct f8mi_gemm_job {
    const void *a, *bt;
    int a_fmt, b_fmt, a_transposed, b_transposed;
    int64_t m, n, k;
    const float *scale_a_dev, *scale_b_dev;
    void* c;
    int64_t ldc;
    int c_dtype;
    void* workspace;
    int64_t workspace_bytes;
} f8mi_gemm_job;

/* Two independent products, as the backward of a linear has them (a: grad_input, b: grad_weight): in one launch where that pays,
 * else one after the other; the same bits.  One launch takes e5m2 times e4m3 with k % 128 == 0 and k >= 384, both pairs of operands as
 * they are, or a with bt transposed and b with both.  tiles: F8MI_PAIR_BY_SIZE, or (for tests and measurements) those of a and of b in one
 * launch, F8MI_PAIR_TILES(a, b), F8MI_ERR_UNSUPPORTED with nothing queued where it does not take them.  The same for a 16-bit result in fp32 that runs on other
 * kernels than tiles. */
#define F8MI_PAIR_BY_SIZE 0
#define F8MI_PAIR_TILES128 1
#define F8MI_PAIR_TILES128X256 2
#define F8MI_PAIR_TILES256 3
#define F8MI_PAIR_TILES(a, b) ((a) | (b) << 2)
int f8mi_gemm_pair(const f8mi_gemm_job* a, const f8mi_gemm_job* b, int tiles, void* stream);

/* f8mi_gemm_nt on ROW-MAJOR fp8 operands either of which may be given transposed, so that the fp8 transposes
 * preprocess_addmm makes for torch._scaled_mm's layout rule (a row-major, b column-major: float8_ops.py:131-155, the
 * .t().contiguous().t() of :150-153) need not be made: the matrix-core kernel transposes on the way from LDS to the
 * registers.
 *   a, a_transposed = 0: [m][k], row stride lda >= k;  = 1: [k][m], row stride lda >= m (the memory of a.t())
 *   bt, b_transposed = 0: [n][k], row stride ldb >= k; = 1: [k][n], row stride ldb >= n (b of a @ b, row-major)
 * In the reference's words: forward x @ W.t() is (0, 0); grad_input dY @ W, W row-major, is (0, 1); grad_weight
 * dY.t() @ x, both row-major, is (1, 1).  (0, 0) is f8mi_gemm_nt.  Transposed operands are taken when k % 128 == 0,
 * k >= 384, the transposed operand's row count (n; m too for (1, 1)) is a multiple of 64, addresses and row strides
 * are 16-byte aligned and the output has more than 256 tiles of 128 x 128; otherwise, and for (1, 0), the call
 * returns F8MI_ERR_UNSUPPORTED without having launched anything and the caller makes the copy the reference makes.
 * Same result bits as f8mi_gemm_nt on the copies. */
int f8mi_gemm_ex(const void* a, int a_fmt, int a_transposed, int64_t lda, const void* bt, int b_fmt, int b_transposed, int64_t ldb,
                 int64_t m, int64_t n, int64_t k, const float* scale_a_dev, const float* scale_b_dev, void* c, int c_dtype,
                 int64_t ldc, const void* bias_dev, void* stream);

/* One (layer, tensor) row of the delayed-scaling bookkeeping; all device pointers. */
typedef struct f8mi_sync_entry {
    float* amax;    /* [1]        fp8_amax_*          */
    float* history; /* [hist_len] fp8_amax_history_*  */
    float* scale;   /* [1]        fp8_scale_*         */
    int64_t fp8_fmt;
} f8mi_sync_entry;

/*
 * For each of the n entries: S = roll(history, 1); S[0] = amax;
 * scale = fmax * (1 / clamp(max(S), 1e-12)) in fp32 (<= 65504 if orig_is_fp16).
 * Replaces the body of sync_float8_amax_and_scale_history
 * (float8_linear_utils.py:287-319: _update_history_stack :37-56 and
 * amax_history_to_scale_stack, float8_utils.py:80-99) in one launch.
 * writeback_history = 0 reproduces the reference, which rolls a stacked copy
 * and leaves each layer's history buffer untouched; 1 stores S back.
 * `entries_dev` is a device array of n f8mi_sync_entry.
 */
int f8mi_sync(const f8mi_sync_entry* entries_dev, int n, int hist_len, int orig_is_fp16, int writeback_history,
              void* stream);

/* f8mi_sync with the entries in HOST memory: they travel to the GPU by value, as kernel arguments, 32 per launch, so
 * there is no table in device memory to build, copy or keep alive.  For callers whose device allocations are managed
 * by someone else -- a compiled graph under torch.compile(mode="reduce-overhead") must not keep a tensor of its own
 * inside the graph's memory pool -- and for one-off calls.  Under stream capture the pointers are baked into the
 * captured launches: the buffers must stay where they are (as for any captured kernel). */
int f8mi_sync_host(const f8mi_sync_entry* entries_host, int n, int hist_len, int orig_is_fp16, int writeback_history,
                   void* stream);

/*
 * First-iteration initialisation of one tensor's buffers
 * (_maybe_initialize_amaxes_scales_for_float8_cast, float8_scaling_utils.py:99-125):
 * history[0] = *amax; *scale = fmax * (1 / clamp(max(history), 1e-12)).
 * `amax_dev` must already hold this step's amax (f8mi_amax_scale).
 */
int f8mi_delayed_init(const float* amax_dev, float* history_dev, float* scale_dev, int hist_len, int fp8_fmt,
                      int orig_is_fp16, void* stream);

/*
 * Optional per-kernel timing with HIP events on the launch stream.  While
 * enabled every launch of kernel class `kernel` (F8MI_K_*) is bracketed by two
 * events; f8mi_prof_read synchronises them and returns launches, summed
 * milliseconds and summed algorithmic work (bytes for amax/cast/sync, flop for
 * gemm).  Off by default; meant for benchmarks, not for training loops.
 */
int f8mi_prof_enable(int on);
int f8mi_prof_reset(void);
int f8mi_prof_read(int kernel, uint64_t* launches, double* total_ms, double* total_work);

#ifdef __cplusplus
}
#endif
#endif /* F8MI_H */
