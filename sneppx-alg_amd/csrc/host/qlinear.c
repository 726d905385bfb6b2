/*
 * qlinear.c - device-pointer entry points (include/sneppx_qlinear.h):
 * argument checks, shape dispatch and workspace, then the HIP launchers.
 * Nothing here touches tensor data; every call is asynchronous on `stream`.
 */
#include <stdint.h>
#include <stdlib.h>

#include "sneppx_qlinear.h"
#include "snx_hip.h"
#include "../snx_internal.h"

/* rows from which W4A16 may run the prefill GEMM with an fp32 result: its
 * fp32 sums are 2e-6 off where the batch kernel's are 1e-7 and those of the
 * GEMVs before it 1e-6.  A bf16 result hides either; it may run the GEMM
 * from half a row tile on. */
#define SNX_W4_GEMM_MIN_M 256
#define SNX_W4_GEMM_MIN_M_BF16 64

static int aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

#define REQUIRE(cond, ...)               \
    do {                                 \
        if (!(cond)) {                   \
            snx_set_error(__VA_ARGS__);  \
            return -1;                   \
        }                                \
    } while (0)

int SNEPPX_dev_quantize_int8_channel(const float* in, int8_t* q, float* scales, size_t rows,
                                     size_t cols, SNEPPXStream stream) {
    REQUIRE(in && q && scales, "dev_quantize_int8_channel: NULL pointer");
    REQUIRE(rows && cols, "dev_quantize_int8_channel: empty matrix");
    snx_clear_error();
    return snx_k_quant_int8_rows(in, q, scales, rows, cols, 0, stream);
}

int SNEPPX_dev_quantize_int8_channel_rounding(const float* in, int8_t* q, float* scales,
                                              size_t rows, size_t cols, SNEPPXRounding rounding,
                                              SNEPPXStream stream) {
    REQUIRE(in && q && scales, "dev_quantize_int8_channel_rounding: NULL pointer");
    REQUIRE(rows && cols, "dev_quantize_int8_channel_rounding: empty matrix");
    REQUIRE(rounding == SNEPPX_ROUND_HALF_AWAY || rounding == SNEPPX_ROUND_HALF_EVEN,
            "dev_quantize_int8_channel_rounding: unknown rounding %d", (int)rounding);
    snx_clear_error();
    return snx_k_quant_int8_rows(in, q, scales, rows, cols, rounding == SNEPPX_ROUND_HALF_EVEN,
                                 stream);
}

int SNEPPX_dev_fake_quant(const float* in, float* out, size_t n, float scale, int bits,
                          SNEPPXStream stream) {
    REQUIRE(in && out, "dev_fake_quant: NULL pointer");
    REQUIRE(scale > 0.0f, "dev_fake_quant: scale must be > 0");
    REQUIRE(bits >= 2 && bits <= 16, "dev_fake_quant: bits=%d outside [2, 16]", bits);
    snx_clear_error();
    if (n == 0) return 0;
    return snx_k_fake_quant(in, out, n, scale, bits, stream);
}

int SNEPPX_dev_quantize_w4_awq(const float* w, uint32_t* qweight, uint16_t* scales,
                               uint32_t* qzeros, size_t N, size_t K, int group,
                               SNEPPXStream stream) {
    REQUIRE(w && qweight && scales && qzeros, "dev_quantize_w4_awq: NULL pointer");
    REQUIRE(N && K, "dev_quantize_w4_awq: empty matrix");
    REQUIRE(group > 0 && group % 8 == 0 && K % (size_t)group == 0,
            "dev_quantize_w4_awq: group %d must be a positive multiple of 8 dividing K=%zu",
            group, K);
    snx_clear_error();
    return snx_k_w4_awq_quantize(w, qweight, scales, qzeros, N, K, group, stream);
}

/* g_idx is checked on the host (one small copy) so the kernel's LDS indexing
 * by group stays in bounds. */
int SNEPPX_dev_quantize_w4_gptq(const float* w, const int32_t* g_idx, size_t G,
                                uint32_t* qweight, uint16_t* scales, size_t N, size_t K,
                                SNEPPXStream stream) {
    REQUIRE(w && g_idx && qweight && scales, "dev_quantize_w4_gptq: NULL pointer");
    REQUIRE(N && K && G, "dev_quantize_w4_gptq: empty shape");
    REQUIRE(K % 8 == 0, "dev_quantize_w4_gptq: K=%zu must be a multiple of 8", K);
    snx_clear_error();
    int32_t* h = (int32_t*)malloc(K * sizeof(int32_t));
    REQUIRE(h, "dev_quantize_w4_gptq: out of host memory");
    int rc = snx_hip_memcpy_d2h(h, g_idx, K * sizeof(int32_t), stream);
    if (rc == 0) rc = snx_hip_stream_sync(stream);
    for (size_t k = 0; rc == 0 && k < K; k++)
        if (h[k] < 0 || (size_t)h[k] >= G) {
            snx_set_error("dev_quantize_w4_gptq: g_idx[%zu]=%d outside [0, %zu)", k, h[k], G);
            rc = -1;
        }
    free(h);
    if (rc) return -1;
    return snx_k_w4_gptq_quantize(w, g_idx, G, qweight, scales, N, K, stream);
}

int SNEPPX_dev_quantize_fp8_e4m3_scaled(const float* in, uint8_t* out, float* scale_out,
                                        size_t n, SNEPPXStream stream) {
    REQUIRE(in && out && scale_out, "dev_quantize_fp8_e4m3_scaled: NULL pointer");
    REQUIRE(n, "dev_quantize_fp8_e4m3_scaled: n == 0");
    snx_clear_error();
    int parts = snx_reduce_parts(n);
    float* ws = (float*)snx_workspace(((size_t)parts * 2 + 64) * sizeof(float), 0, stream);
    if (!ws) return -1;
    float* rec = ws + (size_t)parts * 2;
    rec = (float*)(((uintptr_t)rec + 15u) & ~(uintptr_t)15u);
    int rc = snx_k_absmax(in, n, ws, parts, stream);
    if (!rc) rc = snx_k_finalize_scale(ws, parts, SNX_SCALE_FP8_240, in, rec, scale_out, stream);
    if (!rc) rc = snx_k_fp8_encode(in, out, n, 0, rec, stream);
    return rc;
}

int SNEPPX_qlinear_w8_gemv(const float* x, const int8_t* qweight, const float* scales,
                           const float* bias, float* y, size_t M, size_t N, size_t K,
                           SNEPPXStream stream) {
    REQUIRE(x && qweight && scales && y, "qlinear_w8_gemv: NULL pointer");
    REQUIRE(M && N && K, "qlinear_w8_gemv: empty shape");
    REQUIRE(K % 16 != 0 || (aligned16(x) && aligned16(qweight)),
            "qlinear_w8_gemv: x and qweight must be 16-byte aligned");
    snx_clear_error();
    if (snx_w8_batch_ok(M, N, K, qweight) && !snx_stream_capturing(stream)) {
        const int splits = snx_w8_batch_splits(M, N, K);
        void* xp = snx_workspace(snx_w8_batch_xp_bytes(M, K), 1, stream);
        void* part = NULL;
        uint32_t* cnt = NULL;
        if (!xp) return -1;
        if (splits > 1 && snx_span_workspaces(snx_w8_batch_part_bytes(M, N, splits), snx_w8_batch_cnt_bytes(M, N),
                                              stream, &part, &cnt))
            return -1;
        return snx_k_w8_batch(x, qweight, scales, y, bias, M, N, K, splits, xp, part, cnt, stream);
    }
    return snx_k_w8_gemv(x, qweight, scales, y, bias, M, N, K, stream);
}

/* Scratch of one W4A16 call: the calling thread's workspace on `stream`, or
 * for the allocation-free entry point the library's static device array
 * (NULL, with the error text set, when the call needs more than it holds). */
static void* w4_scratch(size_t bytes, int noalloc, SNEPPXStream stream) {
    return noalloc ? snx_noalloc_scratch(bytes, "qlinear_w4a16_noalloc")
                   : snx_workspace(bytes, 1, stream);
}

/* The batch kernel with its scratch; glu: N gate/up pairs (see snx_k_w4a16_batch). */
static int w4_batch(const char* who, int noalloc, const uint16_t* x, const uint32_t* qweight, const uint16_t* scales,
                    const uint32_t* qzeros, const float* bias, void* y, int y_f32, size_t M, size_t N, size_t K,
                    int group, int glu, SNEPPXStream stream) {
    const size_t rows = glu ? 2 * N : N;
    const int splits = snx_w4a16_batch_splits(M, rows, K);
    void* part = NULL;
    uint32_t* cnt = NULL;
    if (splits > 1) {
        const size_t pb = snx_w4a16_batch_part_bytes(M, rows, splits), cb = snx_w4a16_batch_cnt_bytes(M, rows);
        if (!noalloc) {
            if (snx_span_workspaces(pb, cb, stream, &part, &cnt)) return -1;
        } else {
            part = snx_noalloc_scratch(pb, who);
            cnt = (uint32_t*)snx_noalloc_counters(cb, who);
            if (!part || !cnt) return -1;
        }
    }
    return snx_k_w4a16_batch(x, qweight, scales, qzeros, y, bias, y_f32, M, N, K, group, glu, splits, part, cnt,
                             stream);
}

/* scratch of the prefill GEMM's activation pass: prepared rows, step sums */
static size_t w4_prep_bytes(size_t M, size_t K) {
    return ((M * K * sizeof(uint16_t) + 255) & ~(size_t)255) + (K / 128) * snx_w4_prep_rows(M) * sizeof(float);
}

/* Whether M x N x K runs the prefill GEMM (whole_k: not in spans of K, as its
 * SwiGLU form and the allocation-free entry point run it): where it may and the
 * batch kernel is not estimated to be faster by a tenth (what the estimates are
 * off by).  N = 4096, K = 14336, M = 193: 66 us in spans, 173 whole-K, the batch
 * kernel 66.
 * Below SNX_W4_GEMM_MIN_M only where the allocation-free entry point has the
 * scratch for it, and with K in whole 512s: the GEMM gives NaN where an infinite
 * activation makes the result infinite, as the decode GEMV of those shapes does,
 * and the batch kernel does not.
 * recorded: the call is captured into a graph and neither the batch kernel nor a
 * smaller GEMM is a choice. */
static int w4_takes_gemm(size_t M, size_t N, size_t K, int group, const uint16_t* scales, const uint32_t* qzeros,
                         int y_f32, int whole_k, int recorded) {
    if (M < (y_f32 || recorded ? SNX_W4_GEMM_MIN_M : SNX_W4_GEMM_MIN_M_BF16) || ((uintptr_t)scales & 3u) != 0 ||
        ((uintptr_t)qzeros & 3u) != 0 || !snx_w4a16_gemm_ok(M, N, K, group) ||
        (M < SNX_W4_GEMM_MIN_M &&
         (w4_prep_bytes(M, K) > SNEPPX_NOALLOC_SCRATCH_BYTES || !snx_w4a16_gemv_supported(64, N, K, group))))
        return 0;
    return recorded || !snx_w4a16_batch_ok(M, N, K, group, scales, qzeros) ||
           10 * snx_w4a16_gemm_cost(M, N, K, whole_k ? 1 : snx_w4a16_gemm_splits(M, N, K)) <= 11 * snx_w4a16_batch_cost(M, N, K);
}

/* One row, and M <= 4 within the LDS-staged small-M kernel (groups of 256 and
 * more): 7.3 and 8.1 us at M = 1, 2 (N = 6144, K = 4096), the batch kernel
 * 9.4; stacked gate/up rows and their SwiGLU at M = 1, F = 1408, K = 1792: 5.1
 * and 8.2. */
static int w4_small(size_t M, size_t K, int group, const uint16_t* scales, const uint32_t* qzeros) {
    return M == 1 ? snx_w4a16_gemv1_ok(1, K, group, scales, qzeros) || snx_w4a16_small_ok(1, K, group, 0)
                  : M <= 4 && snx_w4a16_small_ok(M, K, group, 0);
}

/* Shapes with little to stream, where the start and the meeting of the batch
 * kernel's spans weigh most (us of the other kernel / the batch kernel).
 * 17 rows and more, the decode GEMV, while its workgroups of 16 columns are few:
 *   M = 17, 32, K = 512: N = 4096 - , 4.3 / 5.0; 6144 4.2 / 4.8, 4.8 / 4.9;
 *                        8192 4.3 / 4.8, 4.9 / 5.0; 10240 5.1 / 4.9, 6.0 / 4.9
 *   K = 1024:            N = 4096 - , 6.1 / 7.6; 6144 5.8 / 7.2, 7.0 / 7.4;
 *                        8192 5.9 / 7.3, 7.0 / 7.4; 10240 7.0 / 7.6, 9.1 / 7.5
 *   K = 1536:            N = 4096 6.6 / 7.7, 7.5 / 7.7; 8192 7.6 / 8.1, 9.3 / 8.3
 *   K = 2048, N = 4096:  M = 17 7.9 / 8.5, 28 8.2 / 8.5, 32 8.6 / 8.5
 *   M = 33, 48, 64, K = 512: N = 4096 5.3 / 6.2, 5.7 / 6.3, 6.3 / 6.3 (fp32 5.9 / 6.4);
 *                        8192 5.8 / 6.3, 6.3 / 6.3, 7.5 / 6.3
 *   K = 1024:            N = 4096 7.4 / 8.3, 7.8 / 8.3, 9.0 / 8.4; 6144 8.6 / 8.6
 * 2 to 16 rows, split-K in few spans: K = 7168, N = 512 9.8 / 9.5, 1024 10.0 / 10.6,
 * 2048 10.0 / 10.9, 2560 11.9 / 11.5; K = 8192, N = 1408 11.2 / 12.7, 2048 10.7 / 12.2,
 * 2560 13.4 / 12.5; K = 9216, N = 2048 12.4 / 12.4; N = 961, K = 13312 12.3 / 13.4 (in
 * spans of 256, K = 11008: 23.4 / 12.8).
 * glu: stacked gate/up rows, where the other kernel needs the rule's own pass:
 * K = 512, N = 4096 6.0 / 5.0, but K = 1024 7.0 / 7.5, K = 10240, N = 1536 12.7 / 13.9. */
static int w4_short(size_t M, size_t N, size_t K, int group, int glu) {
    if (M > 16) {
        if (!snx_w4a16_gemv_supported(M < 64 ? M : 64, N, K, group)) return 0;
        if (glu) return M <= 32 && K <= 1024 && N <= 4096;
        if (M <= 19 && N <= (K <= 1024 ? 10240u : K <= 1536 ? 8192u : 4096u) && K <= 2048) return 1;
        if (M <= 32) return N <= 8192 && (K <= 1024 || (N <= 4096 && (K <= 1536 || (K <= 2048 && M <= 28))));
        return (M <= 48 && K <= 1024 && N <= 4096) || (M <= 64 && K <= 512 && N <= (M <= 48 ? 8192u : 4096u));
    }
    if (M < 2 || snx_w4a16_splitk_span(M, K, group) < 512) return 0;
    return (K >= 8192 && N <= 1536) || (!glu && K >= 7168 && K <= 8192 && N >= 1024 && N <= 2048);
}

/* 2 to 16 rows of so many columns that much of the batch kernel's last round of the
 * CUs stays idle: split-K, or the small kernels (M = 8, K = 5120: N = 36864 36 / 52
 * us, 49152 45 / 54, 65536 58 / 56; stacked gate/up rows of K = 8192, F = 20480 69 /
 * 80, 28672 93 / 83). */
static int w4_uneven(size_t M, size_t N, size_t K, int group) {
    return M >= 2 && M <= 16 &&
           (snx_w4a16_splitk_span(M, K, group) >= 512 || snx_w4a16_small_ok(M, K, group, 0)) &&
           snx_w4a16_batch_uneven(M, N);
}

/* SwiGLU blocks whose projection runs the persistent kernel or the small one, in
 * fp32 rows and the rule's own pass, where those two launches take less than the
 * batch kernel's one (us of both / the batch kernel).
 * Persistent kernel, 9 to 16 rows (up to 8 always: 20.8 / 22.5 at F = 14336):
 *   K = 1024: F = 256 6.0 / 6.5, 5504 6.4 / 7.3, 6144 6.6 / 7.4, 6656 7.7 / 7.5
 *   K = 2048: F = 4096 9.1 / 8.5 (M = 9 8.2 / 8.4), 5504 9.0 / 10.1, 6144 9.3 / 10.2,
 *             6656 11.0 / 10.2, 16384 17.4 / 12.4, 20480 20.4 / 21.6, 24576 23.6 / 21.8
 *   K = 3072: F = 5504 9.6 / 12.5, 12288 15.6 / 16.2, 13312 17.4 / 16.4, 17408 21 / 29,
 *             28672 31 / 35
 *   K = 4096: F = 5504 10.7 / 14.5, 14336 19.9 / 21.4, 14848 21.6 / 21.6, 18432 24 / 41,
 *             28672 36 / 44
 * (past F = 16384 the batch kernel's workgroups are more than a round of the CUs).
 * Small kernel at up to 1024 items of 8 activations: M = 2: K = 1536, F = 1792 6.0 /
 * 7.5, 3584 7.2 / 7.6, 5504 8.8 / 8.6; K = 2560, F = 5504 10.4 / 11.2, 11008 14.6 /
 * 13.5; K = 3584, F = 11008 16.1 / 17.3, 14336 17.8 / 17.7; M = 4: K = 2560, F = 2560
 * 9.8 / 8.3. */
static int w4_glu_rows(size_t M, size_t F, size_t K, int group) {
    if (M == 1) return 0;
    if (snx_w4a16_mt_ok(M, K, group, 0))
        return M <= 8 || (K == 1024   ? F <= 6144
                          : K == 2048 ? (F > 5120 && F <= 6144) || (F > 16384 && F <= 20480) || (M <= 10 && F <= 1024)
                          : K == 3072 ? F <= 12288 || F > 16384
                                      : F <= 14336 || F > 16384);
    return snx_w4a16_small_ok(M, K, group, 0) && K >= 1536 && M * K <= 8192 && 4 * F <= 13 * K;
}

/* The scratch that SNEPPX_qlinear_w4a16_noalloc is documented to need:
 * prepared activations from SNX_W4_GEMM_MIN_M rows on, split-K partials for
 * the decode shapes outside the persistent small-M kernel. */
static size_t w4_noalloc_bytes(size_t M, size_t N, size_t K, int group, const uint16_t* scales,
                               const uint32_t* qzeros) {
    const int words = ((uintptr_t)scales & 3u) == 0 && ((uintptr_t)qzeros & 3u) == 0;
    if (M >= SNX_W4_GEMM_MIN_M && words && snx_w4a16_gemm_ok(M, N, K, group)) return w4_prep_bytes(M, K);
    const int kspan = snx_w4a16_splitk_span(M, K, group);
    if (kspan && !(words && snx_w4a16_mt_ok(M, K, group, 0)) &&
        (M > 4 || (M > 1 && !snx_w4a16_small_ok(M, K, group, 0))))
        return K / (size_t)kspan * M * N * sizeof(float);
    return 0;
}

static int w4a16_linear(const char* who, int noalloc, const uint16_t* x, const uint32_t* qweight,
                        const uint16_t* scales, const uint32_t* qzeros, const int32_t* g_idx,
                        size_t G, const float* bias, void* y, SNEPPXDtype y_dtype, size_t M,
                        size_t N, size_t K, int group, SNEPPXStream stream) {
    REQUIRE(x && qweight && scales && y, "%s: NULL pointer", who);
    REQUIRE(M && N && K, "%s: empty shape", who);
    REQUIRE(K % 8 == 0, "%s: K=%zu must be a multiple of 8", who, K);
    REQUIRE(y_dtype == SNEPPX_BFLOAT16 || y_dtype == SNEPPX_FLOAT32,
            "%s: y_dtype must be SNEPPX_BFLOAT16 or SNEPPX_FLOAT32", who);
    int y_f32 = y_dtype == SNEPPX_FLOAT32;
    if (g_idx) {
        REQUIRE(G > 0, "%s: G must be > 0 with g_idx", who);
    } else {
        REQUIRE(group > 0 && K % (size_t)group == 0, "%s: group %d must divide K=%zu", who, group, K);
        G = K / (size_t)group;
    }
    snx_clear_error();
    const int aligned = !g_idx && aligned16(x) && aligned16(qweight);
    /* the allocation-free entry point's limit is the one its header gives, also
     * where the batch kernel would need less */
    if (noalloc && aligned && !snx_noalloc_scratch(w4_noalloc_bytes(M, N, K, group, scales, qzeros), who)) return -1;
    /* (a call of the M = 1 kernels takes no workspace, and is not asked about) */
    const int recorded = !noalloc && !(M == 1 && w4_small(M, K, group, scales, qzeros)) && snx_stream_capturing(stream);
    if (aligned && w4_takes_gemm(M, N, K, group, scales, qzeros, y_f32, noalloc, recorded)) {
        /* prefill GEMM: activations prepared once into the call's scratch */
        const size_t Mp = snx_w4_prep_rows(M);
        const size_t xp_bytes = (M * K * sizeof(uint16_t) + 255) & ~(size_t)255;
        char* ws = (char*)w4_scratch(w4_prep_bytes(M, K), noalloc, stream);
        if (!ws) return -1;
        uint16_t* xp = (uint16_t*)ws;
        float* xs = (float*)(ws + xp_bytes);
        /* with few tiles, K in spans (partials in a workspace; not for the
         * allocation-free entry point) */
        const int splits = noalloc ? 1 : snx_w4a16_gemm_splits(M, N, K);
        void* part = NULL;
        uint32_t* cnt = NULL;
        if (splits > 1 && snx_span_workspaces(snx_w4a16_gemm_part_bytes(M, N, splits), snx_w4a16_gemm_cnt_bytes(M, N),
                                              stream, &part, &cnt))
            return -1;
        int rc = snx_k_w4_prep_x(x, xp, xs, M, K, Mp, stream);
        if (!rc) rc = snx_k_w4a16_gemm(xp, xs, qweight, scales, qzeros, y, bias, y_f32, M, N, K,
                                       group, Mp, splits, part, cnt, stream);
        return rc;
    }
    if (!g_idx && snx_w4a16_mt_ok(M, K, group, 0) && aligned16(x) && aligned16(qweight) &&
        ((uintptr_t)scales & 3u) == 0 && ((uintptr_t)qzeros & 3u) == 0) {
        /* 2 <= M <= 16: one persistent workgroup per CU, activations staged once */
        return snx_k_w4a16_gemv_mt(x, qweight, scales, qzeros, NULL, y, bias, y_f32, M, N, K, stream);
    }
    if (aligned && !recorded && !w4_small(M, K, group, scales, qzeros) && !w4_short(M, N, K, group, 0) &&
        !w4_uneven(M, N, K, group) && snx_w4a16_batch_ok(M, N, K, group, scales, qzeros))
        return w4_batch(who, noalloc, x, qweight, scales, qzeros, bias, y, y_f32, M, N, K, group, 0, stream);
    const int kspan = snx_w4a16_splitk_span(M, K, group);
    if (!g_idx && (M > 4 || (M > 1 && !snx_w4a16_small_ok(M, K, group, 0))) && kspan &&
        aligned16(x) && aligned16(qweight)) {
        /* 5 <= M <= 16, and 2 <= M <= 4 where the LDS-staged small-M kernel does
         * not apply (large K): split-K decode + ordered reduction of the partials */
        const size_t S = K / (size_t)kspan;
        float* part = (float*)w4_scratch(S * M * N * sizeof(float), noalloc, stream);
        if (!part) return -1;
        int rc = snx_k_w4a16_splitk(x, qweight, scales, qzeros, part, M, N, K, group, kspan, stream);
        if (!rc) rc = snx_k_w4a16_reduce(part, y, y_f32, (int)S, M * N, N, bias, stream);
        return rc;
    }
    if (!g_idx && M == 1 && aligned16(x) && aligned16(qweight) &&
        snx_w4a16_gemv1_ok(1, K, group, scales, qzeros))
        /* the streaming M = 1 kernel (K a multiple of 256 up to 16384) */
        return snx_k_w4a16_gemv(x, qweight, scales, qzeros, NULL, y, bias, y_f32, 1, N, K, group, stream);
    if (!g_idx && aligned16(x) && aligned16(qweight) &&
        snx_w4a16_gemv_supported(M < 64 ? M : 64, N, K, group)) {
        /* decode GEMV; larger M in 64-row slices that reuse each weight load */
        size_t ob = y_f32 ? 4 : 2;
        for (size_t m0 = 0; m0 < M; m0 += 64) {
            size_t mm = M - m0 < 64 ? M - m0 : 64;
            if (snx_k_w4a16_gemv(x + m0 * K, qweight, scales, qzeros, NULL,
                                 (char*)y + m0 * N * ob, bias, y_f32, mm, N, K, group, stream))
                return -1;
        }
        return 0;
    }
    return snx_k_w4a16_generic(x, qweight, scales, qzeros, g_idx, G, y, bias, y_f32, M, N, K,
                               group, stream);
}

int SNEPPX_qlinear_w4a16(const uint16_t* x, const uint32_t* qweight, const uint16_t* scales,
                         const uint32_t* qzeros, const int32_t* g_idx, size_t G,
                         const float* bias, void* y, SNEPPXDtype y_dtype, size_t M, size_t N,
                         size_t K, int group, SNEPPXStream stream) {
    return w4a16_linear("qlinear_w4a16", 0, x, qweight, scales, qzeros, g_idx, G, bias, y, y_dtype,
                        M, N, K, group, stream);
}

int SNEPPX_qlinear_w4a16_noalloc(const uint16_t* x, const uint32_t* qweight,
                                 const uint16_t* scales, const uint32_t* qzeros,
                                 const int32_t* g_idx, size_t G, const float* bias, void* y,
                                 SNEPPXDtype y_dtype, size_t M, size_t N, size_t K, int group,
                                 SNEPPXStream stream) {
    return w4a16_linear("qlinear_w4a16_noalloc", 1, x, qweight, scales, qzeros, g_idx, G, bias, y,
                        y_dtype, M, N, K, group, stream);
}

/* Stable counting sort of g_idx on the host (one small copy each way). */
int SNEPPX_qlinear_w4_actorder_prepare(const uint32_t* qweight, const int32_t* g_idx, size_t G,
                                       uint32_t* qweight_sorted, uint16_t* perm, size_t N,
                                       size_t K, SNEPPXStream stream) {
    REQUIRE(qweight && g_idx && qweight_sorted && perm, "w4_actorder_prepare: NULL pointer");
    REQUIRE(N && K && G, "w4_actorder_prepare: empty shape");
    REQUIRE(qweight != qweight_sorted, "w4_actorder_prepare: qweight_sorted must not alias qweight");
    REQUIRE(K % 8 == 0 && K <= 65536, "w4_actorder_prepare: K=%zu must be a multiple of 8 and <= 65536", K);
    REQUIRE(K % G == 0, "w4_actorder_prepare: G=%zu must divide K=%zu", G, K);
    snx_clear_error();
    const size_t per = K / G;
    int32_t* h = (int32_t*)malloc(K * sizeof(int32_t));
    uint16_t* hp = (uint16_t*)malloc(K * sizeof(uint16_t));
    size_t* next = (size_t*)calloc(G, sizeof(size_t));
    int rc = (h && hp && next) ? 0 : -1;
    if (rc) snx_set_error("w4_actorder_prepare: out of host memory");
    if (!rc) rc = snx_hip_memcpy_d2h(h, g_idx, K * sizeof(int32_t), stream);
    if (!rc) rc = snx_hip_stream_sync(stream);
    for (size_t k = 0; !rc && k < K; k++) {
        if (h[k] < 0 || (size_t)h[k] >= G) {
            snx_set_error("w4_actorder_prepare: g_idx[%zu]=%d outside [0, %zu)", k, h[k], G);
            rc = -1;
        } else if (next[h[k]]++ == per) {
            snx_set_error("w4_actorder_prepare: group %d holds more than K/G=%zu columns", h[k], per);
            rc = -1;
        }
    }
    /* every group now holds exactly K/G columns: slot g*per + rank in g */
    for (size_t g = 0; !rc && g < G; g++) next[g] = g * per;
    for (size_t k = 0; !rc && k < K; k++) hp[next[h[k]]++] = (uint16_t)k;
    if (!rc) rc = snx_hip_memcpy_h2d(perm, hp, K * sizeof(uint16_t), stream);
    if (!rc) rc = snx_k_w4_permute_cols(qweight, perm, qweight_sorted, N, K, stream);
    if (!rc) rc = snx_hip_stream_sync(stream);
    free(h);
    free(hp);
    free(next);
    return rc ? -1 : 0;
}

int SNEPPX_qlinear_w4a16_actorder(const uint16_t* x, const uint32_t* qweight_sorted,
                                  const uint16_t* scales, const uint32_t* qzeros,
                                  const uint16_t* perm, const float* bias, void* y,
                                  SNEPPXDtype y_dtype, size_t M, size_t N, size_t K, int group,
                                  SNEPPXStream stream) {
    REQUIRE(x && qweight_sorted && scales && perm && y, "qlinear_w4a16_actorder: NULL pointer");
    REQUIRE(M && N && K, "qlinear_w4a16_actorder: empty shape");
    REQUIRE(K % 8 == 0 && K <= 65536, "qlinear_w4a16_actorder: K=%zu must be a multiple of 8 and <= 65536", K);
    REQUIRE(y_dtype == SNEPPX_BFLOAT16 || y_dtype == SNEPPX_FLOAT32,
            "qlinear_w4a16_actorder: y_dtype must be SNEPPX_BFLOAT16 or SNEPPX_FLOAT32");
    REQUIRE(group > 0 && K % (size_t)group == 0,
            "qlinear_w4a16_actorder: group %d must divide K=%zu", group, K);
    snx_clear_error();
    if (aligned16(x) && aligned16(qweight_sorted) && aligned16(perm) && ((uintptr_t)scales & 3u) == 0 &&
        ((uintptr_t)qzeros & 3u) == 0 && snx_w4a16_mt_ok(M, K, group, 1))
        return snx_k_w4a16_gemv_mt(x, qweight_sorted, scales, qzeros, perm, y, bias,
                                   y_dtype == SNEPPX_FLOAT32, M, N, K, stream);
    if (aligned16(x) && aligned16(qweight_sorted) && aligned16(perm) &&
        (snx_w4a16_small_ok(M, K, group, 1) || snx_w4a16_gemv1_ok(M, K, group, scales, qzeros)))
        return snx_k_w4a16_gemv(x, qweight_sorted, scales, qzeros, perm, y, bias,
                                y_dtype == SNEPPX_FLOAT32, M, N, K, group, stream);
    /* other shapes: gather the activation columns once, then the plain path */
    uint16_t* xs = (uint16_t*)snx_workspace(M * K * sizeof(uint16_t), 0, stream);
    if (!xs) return -1;
    int rc = snx_k_gather_cols(x, perm, xs, M, K, stream);
    if (!rc) rc = SNEPPX_qlinear_w4a16(xs, qweight_sorted, scales, qzeros, NULL, 0, bias, y,
                                       y_dtype, M, N, K, group, stream);
    return rc;
}

int SNEPPX_qlinear_w4a16_swiglu(const uint16_t* x, const uint32_t* qweight,
                                const uint16_t* scales, const uint32_t* qzeros, const float* bias,
                                uint16_t* out, size_t M, size_t F, size_t K, int group,
                                SNEPPXStream stream) {
    REQUIRE(x && qweight && scales && out, "qlinear_w4a16_swiglu: NULL pointer");
    REQUIRE(M && F && K, "qlinear_w4a16_swiglu: empty shape");
    REQUIRE(F % 8 == 0 && K % 8 == 0, "qlinear_w4a16_swiglu: F=%zu and K=%zu must be multiples of 8",
            F, K);
    REQUIRE(group > 0 && K % (size_t)group == 0, "qlinear_w4a16_swiglu: group %d must divide K=%zu",
            group, K);
    REQUIRE(aligned16(out), "qlinear_w4a16_swiglu: out must be 16-byte aligned");
    snx_clear_error();
    const int aligned = aligned16(x) && aligned16(qweight);
    /* one decode row: gate and up rows of an output in one wave, SwiGLU on its total */
    if (M == 1 && aligned && snx_w4a16_gemv1_swiglu_ok(F, K, group, scales, qzeros))
        return snx_k_w4a16_gemv1_swiglu(x, qweight, scales, qzeros, bias, out, F, K, group, stream);
    const int recorded = snx_stream_capturing(stream);
    if (aligned && w4_takes_gemm(M, 2 * F, K, group, scales, qzeros, 0, 1, recorded)) {
        const size_t Mp = snx_w4_prep_rows(M);
        const size_t xp_bytes = (M * K * sizeof(uint16_t) + 255) & ~(size_t)255;
        char* ws = (char*)snx_workspace(w4_prep_bytes(M, K), 1, stream);
        if (!ws) return -1;
        uint16_t* xp = (uint16_t*)ws;
        float* xs = (float*)(ws + xp_bytes);
        int rc = snx_k_w4_prep_x(x, xp, xs, M, K, Mp, stream);
        if (!rc) rc = snx_k_w4a16_gemm_swiglu(xp, xs, qweight, scales, qzeros, out, bias, M, F, K,
                                              group, Mp, stream);
        return rc;
    }
    if (aligned && !recorded && !w4_glu_rows(M, F, K, group) && !(M == 1 && w4_small(M, K, group, scales, qzeros)) &&
        !w4_short(M, 2 * F, K, group, 1) && !w4_uneven(M, 2 * F, K, group) &&
        snx_w4a16_batch_ok(M, 2 * F, K, group, scales, qzeros))
        return w4_batch("qlinear_w4a16_swiglu", 0, x, qweight, scales, qzeros, bias, out, 0, M, F, K, group, 1, stream);
    /* other shapes: the [M][2F] projection in fp32 scratch, then the same rule */
    float* gu = (float*)snx_workspace(M * 2 * F * sizeof(float), 0, stream);
    if (!gu) return -1;
    int rc = SNEPPX_qlinear_w4a16(x, qweight, scales, qzeros, NULL, 0, bias, gu, SNEPPX_FLOAT32, M,
                                  2 * F, K, group, stream);
    if (!rc) rc = snx_k_silu_mul_f32(gu, out, M, F, stream);
    return rc;
}

/* workspace slot of the MLP's SwiGLU rows (prepared or plain) */
#define SLOT_MLP_ACT 6

int SNEPPX_qlinear_w4a16_mlp(const uint16_t* x, const uint32_t* gu_qweight, const uint16_t* gu_scales,
                             const uint32_t* gu_qzeros, const float* gu_bias, const uint32_t* dn_qweight,
                             const uint16_t* dn_scales, const uint32_t* dn_qzeros, const float* dn_bias,
                             void* y, SNEPPXDtype y_dtype, size_t M, size_t H, size_t F, size_t N,
                             int group, SNEPPXStream stream) {
    REQUIRE(x && gu_qweight && gu_scales && dn_qweight && dn_scales && y, "qlinear_w4a16_mlp: NULL pointer");
    REQUIRE(M && H && F && N, "qlinear_w4a16_mlp: empty shape");
    REQUIRE(F % 8 == 0 && H % 8 == 0, "qlinear_w4a16_mlp: F=%zu and H=%zu must be multiples of 8", F, H);
    REQUIRE(group > 0 && H % (size_t)group == 0 && F % (size_t)group == 0,
            "qlinear_w4a16_mlp: group %d must divide H=%zu and F=%zu", group, H, F);
    REQUIRE(y_dtype == SNEPPX_BFLOAT16 || y_dtype == SNEPPX_FLOAT32,
            "qlinear_w4a16_mlp: y_dtype must be SNEPPX_BFLOAT16 or SNEPPX_FLOAT32");
    snx_clear_error();
    const int recorded = M >= SNX_W4_GEMM_MIN_M_BF16 && snx_stream_capturing(stream);
    if (aligned16(x) && aligned16(gu_qweight) && aligned16(dn_qweight) && F % 128 == 0 &&
        w4_takes_gemm(M, 2 * F, H, group, gu_scales, gu_qzeros, 0, 1, recorded) &&
        w4_takes_gemm(M, N, F, group, dn_scales, dn_qzeros, y_dtype == SNEPPX_FLOAT32, 0, recorded)) {
        /* x prepared once; the gate/up GEMM's SwiGLU epilogue writes the down
         * GEMM's prepared input (slot order + step sums) */
        const size_t Mp = snx_w4_prep_rows(M);
        const size_t xp_bytes = (M * H * sizeof(uint16_t) + 255) & ~(size_t)255;
        char* ws = (char*)snx_workspace(xp_bytes + (H / 128) * Mp * sizeof(float), 1, stream);
        const size_t ap_bytes = (M * F * sizeof(uint16_t) + 255) & ~(size_t)255;
        char* wa = (char*)snx_workspace(ap_bytes + (F / 128) * Mp * sizeof(float), SLOT_MLP_ACT, stream);
        if (!ws || !wa) return -1;
        uint16_t* xp = (uint16_t*)ws;
        float* xs = (float*)(ws + xp_bytes);
        uint16_t* ap = (uint16_t*)wa;
        float* as = (float*)(wa + ap_bytes);
        const int splits = snx_w4a16_gemm_splits(M, N, F);
        void* part = NULL;
        uint32_t* cnt = NULL;
        if (splits > 1 && snx_span_workspaces(snx_w4a16_gemm_part_bytes(M, N, splits), snx_w4a16_gemm_cnt_bytes(M, N),
                                              stream, &part, &cnt))
            return -1;
        int rc = snx_k_w4_prep_x(x, xp, xs, M, H, Mp, stream);
        if (!rc) rc = snx_k_w4a16_gemm_swiglu_prep(xp, xs, gu_qweight, gu_scales, gu_qzeros, ap, as, gu_bias,
                                                   M, F, H, group, Mp, stream);
        if (!rc) rc = snx_k_w4a16_gemm(ap, as, dn_qweight, dn_scales, dn_qzeros, y, dn_bias,
                                       y_dtype == SNEPPX_FLOAT32, M, N, F, group, Mp, splits, part, cnt,
                                       stream);
        return rc;
    }
    /* other shapes: the two linears, the SwiGLU rows in a workspace */
    uint16_t* act = (uint16_t*)snx_workspace(M * F * sizeof(uint16_t), SLOT_MLP_ACT, stream);
    if (!act) return -1;
    int rc = SNEPPX_qlinear_w4a16_swiglu(x, gu_qweight, gu_scales, gu_qzeros, gu_bias, act, M, F, H, group,
                                         stream);
    if (!rc) rc = SNEPPX_qlinear_w4a16(act, dn_qweight, dn_scales, dn_qzeros, NULL, 0, dn_bias, y, y_dtype,
                                       M, N, F, group, stream);
    return rc;
}

int SNEPPX_qlinear_silu_mul(const uint16_t* gate_up, uint16_t* out, size_t T, size_t F,
                            SNEPPXStream stream) {
    REQUIRE(gate_up && out, "qlinear_silu_mul: NULL pointer");
    REQUIRE(T && F, "qlinear_silu_mul: empty shape");
    REQUIRE(F % 8 == 0, "qlinear_silu_mul: F=%zu must be a multiple of 8", F);
    REQUIRE(aligned16(gate_up) && aligned16(out), "qlinear_silu_mul: buffers must be 16-byte aligned");
    snx_clear_error();
    return snx_k_silu_mul(gate_up, out, T, F, stream);
}

int SNEPPX_qlinear_silu_mul_quant_int8(const uint16_t* gate_up, int8_t* q, float* scales,
                                       size_t T, size_t F, SNEPPXStream stream) {
    REQUIRE(gate_up && q && scales, "qlinear_silu_mul_quant_int8: NULL pointer");
    REQUIRE(T && F, "qlinear_silu_mul_quant_int8: empty shape");
    REQUIRE(F % 8 == 0 && F <= 32768, "qlinear_silu_mul_quant_int8: F=%zu must be a multiple of 8, <= 32768", F);
    REQUIRE(aligned16(gate_up) && ((uintptr_t)q & 7u) == 0,
            "qlinear_silu_mul_quant_int8: gate_up must be 16-byte and q 8-byte aligned");
    snx_clear_error();
    return snx_k_silu_mul_quant_int8(gate_up, q, scales, T, F, stream);
}

int SNEPPX_dev_quantize_int8_channel_bf16(const uint16_t* in, int8_t* q, float* scales,
                                          size_t rows, size_t cols, SNEPPXStream stream) {
    REQUIRE(in && q && scales, "dev_quantize_int8_channel_bf16: NULL pointer");
    REQUIRE(rows && cols, "dev_quantize_int8_channel_bf16: empty matrix");
    snx_clear_error();
    return snx_k_quant_rows_bf16_fast(in, q, scales, rows, cols, stream);
}

int SNEPPX_qlinear_w8a8_i8(const int8_t* A, const float* sA, const int8_t* W, const float* sW,
                           const float* bias, uint16_t* out, size_t M, size_t N, size_t K,
                           SNEPPXStream stream) {
    REQUIRE(A && sA && W && sW && out, "qlinear_w8a8_i8: NULL pointer");
    REQUIRE(M && N && K, "qlinear_w8a8_i8: empty shape");
    REQUIRE(aligned16(A) && aligned16(W), "qlinear_w8a8_i8: A and W must be 16-byte aligned");
    snx_clear_error();
    return snx_k_i8_gemm(A, W, sA, sW, NULL, out, bias, M, N, K, stream);
}

int SNEPPX_qlinear_i8_gemm_i32(const int8_t* A, const int8_t* W, int32_t* C, size_t M, size_t N,
                               size_t K, SNEPPXStream stream) {
    REQUIRE(A && W && C, "qlinear_i8_gemm_i32: NULL pointer");
    REQUIRE(M && N && K, "qlinear_i8_gemm_i32: empty shape");
    REQUIRE(aligned16(A) && aligned16(W), "qlinear_i8_gemm_i32: A and W must be 16-byte aligned");
    snx_clear_error();
    return snx_k_i8_gemm(A, W, NULL, NULL, C, NULL, NULL, M, N, K, stream);
}

int SNEPPX_qlinear_w8a8_fp8(const uint8_t* A, const float* sA, const uint8_t* W, const float* sW,
                            const float* bias, uint16_t* out, size_t M, size_t N, size_t K,
                            SNEPPXStream stream) {
    REQUIRE(A && sA && W && sW && out, "qlinear_w8a8_fp8: NULL pointer");
    REQUIRE(M && N && K, "qlinear_w8a8_fp8: empty shape");
    REQUIRE(aligned16(A) && aligned16(W), "qlinear_w8a8_fp8: A and W must be 16-byte aligned");
    snx_clear_error();
    return snx_k_fp8_gemm(A, W, sA, sW, out, bias, M, N, K, stream);
}

/* Workspace slot of the dynamically quantized activations (codes, then the
 * per-token scales or the per-tensor scale record at a 256-byte boundary). */
#define SLOT_W8A8_DYN 5

int SNEPPX_qlinear_w8a8_i8_dyn(const uint16_t* A, const int8_t* W, const float* sW,
                               const float* bias, uint16_t* out, size_t M, size_t N, size_t K,
                               SNEPPXStream stream) {
    REQUIRE(A && W && sW && out, "qlinear_w8a8_i8_dyn: NULL pointer");
    REQUIRE(M && N && K, "qlinear_w8a8_i8_dyn: empty shape");
    REQUIRE(aligned16(A) && aligned16(W), "qlinear_w8a8_i8_dyn: A and W must be 16-byte aligned");
    snx_clear_error();
    const size_t qb = (M * K + 255) & ~(size_t)255;
    char* ws = (char*)snx_workspace(qb + M * sizeof(float), SLOT_W8A8_DYN, stream);
    if (!ws) return -1;
    int8_t* aq = (int8_t*)ws;
    float* sa = (float*)(ws + qb);
    int rc = snx_k_quant_rows_bf16_fast(A, aq, sa, M, K, stream);
    if (!rc) rc = snx_k_i8_gemm(aq, W, sa, sW, NULL, out, bias, M, N, K, stream);
    return rc;
}

int SNEPPX_qlinear_w8a8_fp8_dyn(const uint16_t* A, const uint8_t* W, const float* sW,
                                const float* bias, uint16_t* out, size_t M, size_t N, size_t K,
                                SNEPPXStream stream) {
    REQUIRE(A && W && sW && out, "qlinear_w8a8_fp8_dyn: NULL pointer");
    REQUIRE(M && N && K, "qlinear_w8a8_fp8_dyn: empty shape");
    REQUIRE(aligned16(A) && aligned16(W), "qlinear_w8a8_fp8_dyn: A and W must be 16-byte aligned");
    snx_clear_error();
    const size_t n = M * K, qb = (n + 255) & ~(size_t)255;
    const int parts = snx_reduce_parts(n);
    char* ws = (char*)snx_workspace(qb + ((size_t)parts * 2 + 64) * sizeof(float), SLOT_W8A8_DYN, stream);
    if (!ws) return -1;
    uint8_t* aq = (uint8_t*)ws;
    float* part = (float*)(ws + qb);
    float* rec = part + (size_t)parts * 2;
    rec = (float*)(((uintptr_t)rec + 15u) & ~(uintptr_t)15u);
    int rc = snx_k_absmax_bf16(A, n, part, parts, stream);
    /* rec[0] = s_A, the per-tensor scale the GEMM's epilogue multiplies by:
     * the encode kernel reduces the partials itself when it can take the
     * vector path, else a one-block finalize does */
    if (!rc && n % 8 == 0 && ((uintptr_t)aq & 7u) == 0) {
        rc = snx_k_fp8_encode_bf16_pt(A, aq, n, part, parts, rec, stream);
    } else if (!rc) {
        rc = snx_k_finalize_scale(part, parts, SNX_SCALE_FP8_240, NULL, rec, NULL, stream);
        if (!rc) rc = snx_k_fp8_encode_bf16(A, aq, n, rec, stream);
    }
    if (!rc) rc = snx_k_fp8_gemm(aq, W, rec, sW, out, bias, M, N, K, stream);
    return rc;
}
