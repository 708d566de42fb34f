// C ABI of the library (declared in include/dsa_attn.h): argument checks, workspace layout, launches.
#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include <mutex>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include "dsa_common.h"
#include "../../include/dsa_attn.h"

extern "C" {
hipError_t dsa_launch_topk(const float *scores, int64_t ld, int row_begin, int row_end, const int32_t *cu, int N,
                           int K, int32_t *idx, int32_t *n, uint32_t *bitmap, int ldw, float *sel, hipStream_t stream);
hipError_t dsa_launch_indexer_kl(const float *sel, const float *mass, const int32_t *n, int T, int K, float grad_scale,
                                 float *loss, float *dscore, hipStream_t stream);
hipError_t dsa_launch_indexer(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int N,
                              int Hi, int Di, float scale, int row_begin, int row_end, int skip_dense_k,
                              float *scores, int64_t ld, hipStream_t stream);
hipError_t dsa_launch_attn_fwd(const void *q, const void *k, const void *v, const int32_t *idx, const int32_t *n,
                               const int32_t *cu, int N, int T, int Hq, int Hkv, int D, int K, float scale, int pos_min, int split_len,
                               int pos_short, void *out, float *lse, hipStream_t stream);
hipError_t dsa_launch_sel_fwd(const void *q, const void *k, const void *v, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T,
                              int Hq, int Hkv, float scale, int pos_min, int pos_max, int split_len, void *out, float *lse, hipStream_t stream);
hipError_t dsa_launch_sel_dq(const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                             const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float scale, int pos_min,
                             int pos_max, int split_len, void *dq, hipStream_t stream);
hipError_t dsa_launch_selkv(const void *dout, const void *q, const void *k, const void *v, const float *lse, const float *delta,
                            const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T, int Hq, int Hkv, float scale, int split_len,
                            void *dk, void *dv, hipStream_t stream);
hipError_t dsa_launch_delta(const void *dout, const void *out, int T, int Hq, int D, float *delta, hipStream_t stream);
hipError_t dsa_launch_bitmap(const int32_t *idx, const int32_t *n, const int32_t *cu, int N, int T, int K, int ldw,
                             uint32_t *bitmap, hipStream_t stream);
hipError_t dsa_launch_gather_dq(const void *dout, const void *q, const void *k, const void *v, const float *lse,
                                const float *delta, const int32_t *idx, const int32_t *n, const int32_t *cu, int N,
                                int T, int Hq, int Hkv, int D, int K, float scale, int pos_min,
                                int split_len, int pos_short, void *dq, hipStream_t stream);
hipError_t dsa_launch_indexer_bwd(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n, const float *dscore, const float *grad,
                                  const uint32_t *bitmap, int32_t *prefix, float *w_f32, int ldw, const int32_t *cu, int N, int T, int Hi,
                                  int Di, int K, float cscale, void *dq_idx, void *dk_idx, void *dw, int dw_bf16, float *partial,
                                  hipStream_t stream, hipStream_t stream_q);
size_t dsa_indexer_bwd_partial_bytes(int T, int Di, int ldw);
hipError_t dsa_launch_tile_mass(const void *q, const void *k, const float *lse, const uint32_t *bitmap, int ldw,
                                const int32_t *n, const int32_t *cu, int N, int T, int Hq, int Hkv, int D, int K,
                                float scale, float *partial, float *mass, hipStream_t stream);
hipError_t dsa_launch_tile_fwd(const void *q, const void *k, const void *v, const int64_t *strides, const uint32_t *bitmap, int ldw,
                               const int32_t *cu, int N, int T, int Hq, int Hkv, int D, float scale, int pos_split, int split_len,
                               int pos_short, int window, int carried, int causal, void *out, float *lse, hipStream_t stream);
hipError_t dsa_launch_tile_dq(const void *dout, const void *q, const void *k, const void *v, const float *lse,
                              const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T,
                              int Hq, int Hkv, int D, float scale, int pos_split, int split_len, int pos_short, int window, int carried, int causal,
                              void *dq, const void *out_for_delta,
                              float *delta_out, hipStream_t stream);
hipError_t dsa_launch_tile_dkv(const void *dout, const void *q, const void *k, const void *v, const float *lse,
                               const float *delta, const uint32_t *bitmap, int ldw, const int32_t *cu, int N, int T,
                               int Hq, int Hkv, int D, float scale, int carried, int causal, int skip_len, int32_t *order, int listed, float *partial,
                               size_t partial_bytes, void *dk, void *dv, const DqBeside *beside, hipStream_t stream);
hipError_t dsa_launch_tile_order_delta(const void *dout, const void *out, const int32_t *cu, int N, int T, int Hq, int Hkv, int D,
                                       int has_idx, int causal, int32_t *order, const float *partial, size_t partial_bytes,
                                       float *delta, hipStream_t stream);
size_t dsa_tile_order_bytes(int T);
size_t dsa_tile_dkv_partial_bytes(int T);
int dsa_mass_groups(int Hq, int Hkv, int D);
}

extern "C" {
int dsa_prologue_bwd_blocks(int T);
hipError_t dsa_launch_qk_norm_rope_fwd(const void *q_in, int64_t q_tok, int64_t q_head, const void *k_in, int64_t k_tok,
                                       int64_t k_head, const void *qw, const void *kw, int w_bf16, float eps, float w_offset,
                                       const void *cosp, const void *sinp, int cs_f32, int R, int T, int Hq, int Hkv, int D,
                                       void *q_out, void *k_out, float *q_rstd, float *k_rstd, hipStream_t stream);
hipError_t dsa_launch_qk_norm_rope_bwd(const void *gq, const void *gk, const void *q_in, int64_t q_tok, int64_t q_head,
                                       const void *k_in, int64_t k_tok, int64_t k_head, const void *qw, const void *kw,
                                       int w_bf16, float w_offset, const void *cosp, const void *sinp, int cs_f32, int R,
                                       const float *q_rstd, const float *k_rstd, int T, int Hq, int Hkv, int D, void *dq_in,
                                       int64_t dq_tok, int64_t dq_head, void *dk_in, int64_t dk_tok, int64_t dk_head,
                                       void *dqw, void *dkw, int grad_bf16, float *part, hipStream_t stream);
hipError_t dsa_launch_sigmoid_gate_fwd(const void *x, const void *gate, int64_t gate_tok, int64_t gate_head, int D, int H,
                                       int64_t rows, void *y, hipStream_t stream);
hipError_t dsa_launch_pack_columns(int n, const void *const *src, const int32_t *width, const int32_t *group, const int32_t *dst_col,
                                   const int32_t *dst_group, int T, void *dst, int64_t dst_row, hipStream_t stream);
hipError_t dsa_launch_split_stack(const float *x, int64_t rows, int D, int order, void *y, hipStream_t stream);
hipError_t dsa_launch_split_combine(const void *y, int64_t rows, int D, int part, float *out, hipStream_t stream);
hipError_t dsa_launch_round_bf16_x3(const float *a, const float *b, const float *c, int64_t na, int64_t nb, int64_t nc, void *ya,
                                    void *yb, void *yc, hipStream_t stream);
hipError_t dsa_launch_split_stack_qkv(const float *q, const float *k, const float *v, int64_t rows_q, int64_t rows_kv, int D, void *yq,
                                      void *yk, void *yv, hipStream_t stream);
hipError_t dsa_launch_split_combine_qkv(const void *yq, const void *yk, const void *yv, int64_t rows_q, int64_t rows_kv, int D,
                                        float *dq, float *dk, float *dv, hipStream_t stream);
hipError_t dsa_launch_sigmoid_gate_bwd(const void *gy, const void *x, const void *gate, int64_t gate_tok, int64_t gate_head,
                                       int D, int H, int64_t rows, void *dx, void *dgate, int64_t dgate_tok,
                                       int64_t dgate_head, hipStream_t stream);
}

static thread_local char g_err[512] = "";

static int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}
static int hip_fail(hipError_t e, const char *what) {
    return fail(DSA_ERR_HIP, "%s: %s", what, hipGetErrorString(e));
}
static inline size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

#define SCORE_CHUNK_BYTES ((size_t)1 << 30)
static inline int64_t score_ld(int max_seqlen) { return (int64_t)align_up((size_t)max_seqlen, 32); }

extern "C" const char *dsa_version(void) { return "dsa-attn-gfx950 0.1"; }
extern "C" const char *dsa_last_error(void) { return g_err; }

static int check_packed(int T, int N, const int32_t *cu) {
    if (T < 0 || N < 1) return fail(DSA_ERR_ARG, "T=%d N=%d: need T>=0 and at least one segment", T, N);
    if (!cu) return fail(DSA_ERR_ARG, "cu_seqlens is null");
    return DSA_OK;
}

// operands the kernels load straight into LDS, 16 bytes per lane
static int check_aligned(const void *a, const void *b, const char *what) {
    if (((uintptr_t)a | (uintptr_t)b) & 15) return fail(DSA_ERR_ARG, "%s must lie on 16-byte boundaries", what);
    return DSA_OK;
}

extern "C" int dsa_indexer_scores(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int T,
                                  int N, int Hi, int Di, float scale, int dtype, int row_begin, int row_end,
                                  int skip_dense_k, float *scores, int64_t ld, void *stream) {
    if (int rc = check_packed(T, N, cu)) return rc;
    if (dtype != DSA_DTYPE_BF16) return fail(DSA_ERR_UNSUPPORTED, "indexer inputs must be bf16 (dtype code %d)", dtype);
    if (!q_idx || !k_idx || !w_idx || !scores) return fail(DSA_ERR_ARG, "null tensor pointer");
    if (int rc = check_aligned(k_idx, k_idx, "k_idx")) return rc;
    if (row_begin < 0 || row_end > T || row_begin > row_end) return fail(DSA_ERR_ARG, "bad row range [%d,%d)", row_begin, row_end);
    if (Hi < 1 || Hi > 64 || !(Di == 32 || Di == 64 || Di == 128))
        return fail(DSA_ERR_UNSUPPORTED, "indexer geometry Hi=%d Di=%d: need Hi<=64 and Di in {32,64,128}", Hi, Di);
    hipError_t e = dsa_launch_indexer(q_idx, k_idx, w_idx, cu, N, Hi, Di, scale, row_begin, row_end, skip_dense_k,
                                      scores, ld, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "indexer launch");
}

extern "C" int dsa_topk_from_scores(const float *scores, int64_t ld, int row_begin, int row_end, const int32_t *cu,
                                    int T, int N, int K, int32_t *idx, int32_t *n, void *stream) {
    if (int rc = check_packed(T, N, cu)) return rc;
    if (!scores || !idx || !n) return fail(DSA_ERR_ARG, "null tensor pointer");
    if (K < 1) return fail(DSA_ERR_ARG, "top_k=%d must be >= 1", K);
    if (row_begin < 0 || row_end > T || row_begin > row_end) return fail(DSA_ERR_ARG, "bad row range [%d,%d)", row_begin, row_end);
    hipError_t e = dsa_launch_topk(scores, ld, row_begin, row_end, cu, N, K, idx, n, nullptr, 0, nullptr, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "top-k launch");
}

extern "C" size_t dsa_index_topk_workspace_bytes(int T, int max_seqlen, int K) {
    (void)K;
    if (T <= 0 || max_seqlen <= 0) return 0;
    const size_t row_bytes = (size_t)score_ld(max_seqlen) * 4;
    size_t rows = SCORE_CHUNK_BYTES / row_bytes;
    if (rows < 64) rows = 64;
    if (rows > (size_t)T) rows = (size_t)T;
    return align_up(rows, 4) * row_bytes;
}

static inline int bitmap_ldw(int max_seqlen) { return (max_seqlen + 31) / 32; }   // words of a row of the selection bitmap

// sel_scores != NULL: every row is scored (also those whose whole causal window is selected) and the scores of
// the selected keys are kept; bitmap != NULL: the top-k kernel also leaves the inverted selection there
static int index_topk_impl(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int T, int N,
                           int Hi, int Di, int K, float scale, int dtype, int max_seqlen, int32_t *idx, int32_t *n,
                           float *sel_scores, uint32_t *bitmap, void *ws, size_t ws_bytes, void *stream, bool words_only = false) {
    if (int rc = check_packed(T, N, cu)) return rc;
    if (K < 1) return fail(DSA_ERR_ARG, "top_k=%d must be >= 1", K);
    if (max_seqlen < 1 || max_seqlen > T) return fail(DSA_ERR_ARG, "max_seqlen=%d outside [1,T=%d]", max_seqlen, T);
    if ((!idx || !n) && !words_only) return fail(DSA_ERR_ARG, "null output pointer");
    if (T == 0) return DSA_OK;
    const int64_t ld = score_ld(max_seqlen);
    int64_t rows = ws ? (int64_t)(ws_bytes / ((size_t)ld * 4)) : 0;
    rows &= ~(int64_t)3;
    if (max_seqlen <= K && !sel_scores) rows = T;   // every row is dense: no score is read or written
    else if (rows < 4) return fail(DSA_ERR_WORKSPACE, "workspace of %zu bytes holds no score chunk (row = %lld bytes)", ws_bytes, (long long)ld * 4);
    if (rows > T) rows = T;
    for (int64_t r0 = 0; r0 < T; r0 += rows) {
        const int r1 = (int)((r0 + rows < T) ? r0 + rows : T);
        if (max_seqlen > K || sel_scores) {
            int rc = dsa_indexer_scores(q_idx, k_idx, w_idx, cu, T, N, Hi, Di, scale, dtype, (int)r0, r1, sel_scores ? 0 : K,
                                        (float *)ws, ld, stream);
            if (rc) return rc;
        }
        hipError_t e = dsa_launch_topk((const float *)ws, ld, (int)r0, r1, cu, N, K, idx, n, bitmap,
                                       bitmap_ldw(max_seqlen), sel_scores, (hipStream_t)stream);
        if (e != hipSuccess) return hip_fail(e, "top-k launch");
    }
    return DSA_OK;
}

extern "C" int dsa_index_topk(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int T, int N,
                              int Hi, int Di, int K, float scale, int dtype, int max_seqlen, int32_t *idx, int32_t *n,
                              void *ws, size_t ws_bytes, void *stream) {
    return index_topk_impl(q_idx, k_idx, w_idx, cu, T, N, Hi, Di, K, scale, dtype, max_seqlen, idx, n, nullptr, nullptr, ws,
                           ws_bytes, stream);
}

extern "C" int dsa_index_topk_scores(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int T,
                                     int N, int Hi, int Di, int K, float scale, int dtype, int max_seqlen, int32_t *idx,
                                     int32_t *n, float *sel_scores, void *ws, size_t ws_bytes, void *stream) {
    if (!sel_scores) return fail(DSA_ERR_ARG, "null output pointer");
    return index_topk_impl(q_idx, k_idx, w_idx, cu, T, N, Hi, Di, K, scale, dtype, max_seqlen, idx, n, sel_scores, nullptr,
                           ws, ws_bytes, stream);
}

// ---- dsa_index_topk for callers that cannot allocate -------------------------------------------------------
// The score rows live in a file-scope device array instead of a caller's workspace.  Its name is a host-side handle,
// not a device address: the address is looked up once per device (every GPU holds its own copy of the array) and only
// that pointer is ever handed to a kernel.
#define DSA_SCRATCH_BYTES ((size_t)32 << 20)
#define DSA_MAX_DEVICES 64
static __device__ __align__(256) unsigned char scratch[DSA_SCRATCH_BYTES];
static void *g_scratch_ptr[DSA_MAX_DEVICES];
static std::mutex g_scratch_mu;

static int scratch_of_current_device(void **out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= DSA_MAX_DEVICES) return fail(DSA_ERR_UNSUPPORTED, "device %d: the static scratch serves devices 0..%d", dev, DSA_MAX_DEVICES - 1);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return hip_fail(e, "hipGetSymbolAddress(scratch)");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return DSA_OK;
}

extern "C" size_t dsa_index_topk_noalloc_scratch_bytes(void) { return DSA_SCRATCH_BYTES; }
// longest segment whose four score rows (the smallest chunk the chunked loop works on) fit the scratch
extern "C" int dsa_index_topk_noalloc_max_seqlen(void) { return (int)(DSA_SCRATCH_BYTES / (4 * sizeof(float)) / 32 * 32); }

extern "C" int dsa_index_topk_noalloc(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int T,
                                      int N, int Hi, int Di, int K, float scale, int dtype, int max_seqlen, int32_t *idx,
                                      int32_t *n, void *stream) {
    if (max_seqlen > dsa_index_topk_noalloc_max_seqlen())
        return fail(DSA_ERR_WORKSPACE, "max_seqlen=%d: the %zu-byte static scratch holds score rows of at most %d columns; "
                    "use dsa_index_topk with a workspace of your own", max_seqlen, DSA_SCRATCH_BYTES,
                    dsa_index_topk_noalloc_max_seqlen());
    void *ws = nullptr;
    if (int rc = scratch_of_current_device(&ws)) return rc;
    // nothing in the scratch has to start at zero: the indexer writes every column [0, pos] of a row before the
    // selection reads it, and rows whose whole window is selected are never read
    return index_topk_impl(q_idx, k_idx, w_idx, cu, T, N, Hi, Di, K, scale, dtype, max_seqlen, idx, n, nullptr, nullptr, ws,
                           DSA_SCRATCH_BYTES, stream);
}

extern "C" int dsa_indexer_kl(const float *sel_scores, const float *mass, const int32_t *n, int T, int K, float grad_scale,
                              float *loss, float *dscore, void *stream) {
    if (T < 0 || K < 1) return fail(DSA_ERR_ARG, "T=%d, top_k=%d", T, K);
    if (T > 0 && (!sel_scores || !mass || !n || !loss)) return fail(DSA_ERR_ARG, "null tensor pointer");
    hipError_t e = dsa_launch_indexer_kl(sel_scores, mass, n, T, K, grad_scale, loss, dscore, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "indexer KL launch");
}

static int check_attn(int T, int N, const int32_t *cu, int Hq, int Hkv, int D, int K, int dtype, bool selected, const int32_t *idx,
                      const int32_t *n) {
    if (int rc = check_packed(T, N, cu)) return rc;
    if (dtype != DSA_DTYPE_BF16 && !(dtype == DSA_DTYPE_SPLIT_BF16 && D == 256))
        return fail(DSA_ERR_UNSUPPORTED, "q/k/v must be bf16 (dtype code %d)", dtype);
    if (Hq < 1 || Hkv < 1 || Hq % Hkv) return fail(DSA_ERR_ARG, "Hq=%d must be a positive multiple of Hkv=%d", Hq, Hkv);
    if (Hq / Hkv > 16) return fail(DSA_ERR_UNSUPPORTED, "Hq/Hkv=%d: at most 16 query heads per kv head", Hq / Hkv);
    if (!(D == 64 || D == 128 || D == 256 || (D == 96 && !selected)))
        return fail(DSA_ERR_UNSUPPORTED, "head_dim=%d: need 64, 128 or 256 (96 as well without a key selection)", D);
    if ((idx == nullptr) != (n == nullptr)) return fail(DSA_ERR_ARG, "idx and n must both be given or both be null");
    if (selected && K < 1) return fail(DSA_ERR_ARG, "top_k=%d must be >= 1", K);
    if ((int64_t)T * Hkv >= ((int64_t)1 << 31)) return fail(DSA_ERR_UNSUPPORTED, "T*Hkv too large for one launch");
    return DSA_OK;
}

// Query rows whose position in their segment is below top_k * crossover are handled by the tile
// kernels (their selection covers more than 1/crossover of the causal window), the rest by the
// gather kernels.  Process-wide tuning knob; 0 = gather only, a huge value = tile only.
#define DSA_TILE_CROSSOVER 24
static std::atomic<int> g_tile_crossover{DSA_TILE_CROSSOVER};          // read on every launch, possibly from several host threads
extern "C" int dsa_set_tile_crossover(int crossover) {
    if (crossover < 0) return fail(DSA_ERR_ARG, "crossover=%d must be >= 0", crossover);
    g_tile_crossover.store(crossover, std::memory_order_relaxed);
    return DSA_OK;
}
extern "C" int dsa_get_tile_crossover(void) { return g_tile_crossover.load(std::memory_order_relaxed); }

// Who takes a query row, by its position and its segment's length (a segment's own, so that any upper bound of the longest one gives the same
// bits): in segments of at least `len` tokens the tile kernels below `tiles`, the compacted walk (dsa_tile_sel.hip) below `walk`, the gather
// kernels from there on; in shorter ones the tile kernels below `below`, the gather kernels from there on.  Multiples of 256, the coarsest block of
// a tile kernel.
// The compacted walk stands between the other two at head_dim 128 with two to four heads per kv head, unless the crossover was set.  Its rows cost
// what the 32-key steps of their blocks cost, a gathered row what its K keys do, so that the gather is the better one again once rows are long
// (K = 128, 32 768 tokens, two kv heads of 4: forward 0.46 ms gathered, 0.88 walked), the sooner the fewer queries a wave holds.  One
// document, 32 heads over 8 kv heads, K = 2048, gather from 24 K on (tiles up to there) -> walk from 16 K on, forward / backward, ms:
// 131 072 tokens 94.5 / 299 -> 57.3 / 277, 65 536 30.3 / 86.5 -> 21.1 / 78.0, 49 152 16.7 / 49.9 -> 15.0 / 46.8, 40 000 11.2 / 34.2 -> 11.0 / 33.5,
// 36 000 9.1 / 27.7 -> 9.8 / 27.3, 33 000 7.7 / 22.5 -> 8.9 / 23.7.  With 8 and 16 heads per kv head (32 768 tokens, two kv heads, K = 512) the
// gather is the faster one from 16 K on: forward 1.45 and 1.71 ms against 1.84 and 3.29; at head_dim 64 with 4 heads too, 0.59 against 0.81.
// The walk is a launch of its own behind the tiles', as long as its longest row's walk however few the rows are, and the backward forms delta in
// a pass of its own again: it takes rows to win that back.  Operator steps, walk over tiles and gather, 4 to 32 heads of four per kv head, K = 64 to 1024, one segment
// and three, by the rows past 16 K times the heads: 20 000 to 40 000 1.00 to 1.28, 40 000 to 50 000 1.00 to 1.10 (segments of 34 and 40 K 0.96), 50 000 to 60 000 0.93 to
// 1.05, 60 000 to 70 000 0.94 to 1.02, 80 000 to 100 000 0.93 to 1.02, 110 000 to 130 000 0.89 to 0.96.
// Two heads per kv head: a wave holds twice the queries, so that rows have to be thinner, and more of them: 40 000 to 50 000 1.07 to 1.14 (segments of 80 K and more
// 0.94 to 0.98), 60 000 to 80 000 0.99 to 1.07, 90 000 to 100 000 1.00 to 1.05, 100 000 to 120 000 0.94 to 1.02, 140 000 0.91 to 1.01.  The gather, which reads a key's rows for two
// heads, is slower than the tiles wherever the walk does not stand (36 K: 1558 and 1750 us, 70 K: 2696 and 2824).
// A batch without rows for the gather is spared two launches and the selection's list: segments that pass 24 K by less than a third stay on the tiles
// (tile_rows_end), and in batches whose longer ones are walked, from 48 K on at the latest, all shorter ones.  Steps, us, gather from 24 K -> tiles:
// 12 heads over 4, K = 64, 1607 tokens 173 -> 147, 32 over 8 with segments of 31 K and 6 K 316 -> 278, K = 128, 28 K 0.96 on average; from K = 512 on level.
// Beyond, 34 K: 4 over 1, K = 64, 162 -> 180, K = 128 340 -> 374.
#define DSA_WALK_ROWS 48000                              // rows times heads (of groups padded to a power of two), at least
#define DSA_WALK_ROWS_2 100000                           // with two heads per kv head,
#define DSA_WALK_ROWS_2_LONG 40000                       // of segments that pass the tiles
struct RowSplit {
    int tiles, walk, len, below;
    bool walks(int max_seqlen) const { return walk > tiles && max_seqlen > tiles && max_seqlen >= len; }
    // (the only segment of a batch has all of its tokens)
    bool gathers(int max_seqlen, int T, int N) const {
        return (max_seqlen > walk && max_seqlen >= len) || (max_seqlen < len ? tile_rows_end(max_seqlen, tiles, len, below) < max_seqlen
                                                                             : tile_rows_end(len - 1, tiles, len, below) < len - 1 && (N != 1 || T < len));
    }
};
// (N = 0: of a segment whose batch is not known, which takes no fewer rows to walk than any batch)
static RowSplit row_split_for(bool selected, const int32_t *idx, int T, int N, int Hq, int Hkv, int D, int K) {
    if (!selected) return {INT32_MAX, INT32_MAX, 0, INT32_MAX};           // dense causal: tiles everywhere
    auto line = [&](int64_t times) {
        const int64_t p = K * times;
        return p >= INT32_MAX - 256 ? INT32_MAX : (int)((p + 255) / 256 * 256);
    };
    const int crossover = g_tile_crossover.load(std::memory_order_relaxed), G = Hq / Hkv;
    const bool two = G == 2;
    if (crossover != DSA_TILE_CROSSOVER || D != 128 || G < 2 || G > 4) {
        const int split = idx ? line(crossover) : INT32_MAX;
        return {split, split, 0, split};
    }
    // tokens of a segment that has `rows` by itself, or, where the segments of the batch are long on average, with as many like it as there are tokens for
    const int heads = Hkv << (two ? 1 : 2), least = line(two ? 26 : 18);
    const double all = (double)T * heads;
    auto len_for = [&](double rows) {
        auto past = [&](double more) { return std::max(least, (int)std::min(16. * K + more, (double)INT32_MAX)); };
        const int alone = past(rows / heads), many = all > rows ? past(16. * K * rows / (all - rows)) : INT32_MAX;
        return N > 0 && T / N >= many ? std::min(many, alone) : alone;
    };
    RowSplit s{line(16), line(two ? 150 : 75), len_for(two ? DSA_WALK_ROWS_2 : DSA_WALK_ROWS), line(two ? 75 : crossover)};
    if (two && s.len > s.below) s.len = std::min(s.len, std::max(s.below + 1, len_for(DSA_WALK_ROWS_2_LONG)));
    if (s.len > s.walk) s = {s.below, s.below, INT32_MAX, s.below};       // (rows too thin for the walk before there are enough of them)
    else if (N > 1 && s.len <= line(48)) s.below = std::max(s.below, s.len - 1);
    if (!idx) s = {s.tiles, INT32_MAX, s.len, INT32_MAX};                 // no list to gather by
    return s;
}
extern "C" int dsa_attn_reads_list(int Hq, int Hkv, int D, int K, int max_seqlen) {
    if (Hkv < 1 || Hq < Hkv || K < 1) return 1;
    static const int32_t some = 0;
    return row_split_for(true, &some, 0, 0, Hq, Hkv, D, K).gathers(max_seqlen, 0, 0);
}
extern "C" int dsa_attn_batch_reads_list(int Hq, int Hkv, int D, int K, int T, int N, int max_seqlen) {
    if (Hkv < 1 || Hq < Hkv || K < 1) return 1;
    static const int32_t some = 0;
    return row_split_for(true, &some, T, N, Hq, Hkv, D, K).gathers(max_seqlen, T, N);
}

// The key side of segments of at least this many tokens is the compacted walk's (dsa_tile_selkv.hip) rather than the tile kernel's: head_dim 128,
// three and more heads per kv head, launches that the tile kernel does not cut into pieces (its workgroups, 192 keys each, are cut nowhere: four
// rounds of them end level).  A walk pays for building the list of every block of queries, and adds the rounding remainder of P to dV where a step
// has a probability of 2^-7, the tile kernel where a block has one of 2^-6: up to some hundred keys a row both do nearly always, with flat rows of
// 128 to some 200 the walk alone.  dK and dV alone, walk over tile kernel, random scores, 30 000 / 56 000 tokens in all, 32 heads over 8 (24 over 8 the same):
// K = 32: segments of 33 K 1.00 / 0.91, 40 K 0.96 / 0.87; K = 64: 33 K 1.06 / 0.99, 36 K 0.91 / 0.85, 60 K 0.74 / 0.70; K = 96: 28 K 1.00 / 0.93, 40 K 0.86 / 0.82;
// K = 128: 36 K 1.13 / 1.03, 45 K 1.11 / 1.00, 52 K 0.98 / 0.93; K = 192: 40 K 1.07, 52 K 0.99 / 0.94; K = 256: 30 K 1.06, 33 K 1.01 / 1.00, 40 K 0.91; K = 512: 24 K 1.02 / 1.06,
// 30 K 1.00, 40 K 0.87; K = 1024: 24 K 0.98 / 1.05, 28 K 1.02, 36 K 0.92.  64 over 16: K = 128, 36 K 1.01, 45 K 0.91; K = 256, 36 K 0.95.  With fewer kv heads
// it pays later: 16 over 4, 56 000 tokens: K = 64, 45 K 1.08, 60 K 0.78; K = 128, 60 K 1.02; K = 256, 36 K 1.09; K = 512, 36 K 0.93.  Whole backward, ms,
// 32 over 8, K = 2048: 40 000 tokens 34.0 -> 35.5, 49 152 47.5 -> 48.5, 57 344 63.3 -> 61.7, 65 536 79.5 -> 75.8, 81 920 117.9 -> 106.6, 131 072 281 -> 226.
static int key_walk_len(bool selected, const void *q, const void *dout, int T, int N, int Hq, int Hkv, int D, int K) {
    const int G = Hq / Hkv;
    if (!selected || D != 128 || G < 3 || ((int64_t)T / 128 + N) * Hkv <= dkv_pieces_max_wg(D) || (((uintptr_t)q | (uintptr_t)dout) & 15) ||
        g_tile_crossover.load(std::memory_order_relaxed) != DSA_TILE_CROSSOVER)
        return INT32_MAX;
    const int64_t len = K <= 112 ? K * 40ll : K < 256 ? K * 50ll : K * 24ll + 3072;
    return (int)std::min<int64_t>(Hkv < 8 ? len * 6 / 5 : len, INT32_MAX);
}

extern "C" size_t dsa_attn_fwd_workspace_bytes(int T, int max_seqlen, int has_idx) {
    if (T <= 0 || !has_idx) return 0;
    return align_up((size_t)T * bitmap_ldw(max_seqlen) * 4, 256);
}

// idx null with `selected`: ws holds a bitmap that a selection of K keys per row left, so that rows at positions below K attend all of their window
// build_bitmap == 0: ws already holds the bitmap of idx/n (it is only read)
static int attn_fwd_run(const void *q, const void *k, const void *v, bool selected, const int32_t *idx, const int32_t *n, const int32_t *cu,
                        int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale, int dtype, int max_seqlen, int causal,
                        void *out, float *lse, void *ws, size_t ws_bytes, int build_bitmap, void *stream) {
    if (int rc = check_attn(T, N, cu, Hq, Hkv, D, K, dtype, selected, idx, n)) return rc;
    if (!causal && selected) return fail(DSA_ERR_ARG, "a key selection (idx) implies causal attention");
    if (!q || !k || !v || !out || !lse) return fail(DSA_ERR_ARG, "null tensor pointer");
    if (int rc = check_aligned(k, v, "k and v")) return rc;
    if (max_seqlen < 1 || max_seqlen > (T > 0 ? T : 1)) return fail(DSA_ERR_ARG, "max_seqlen=%d outside [1,T=%d]", max_seqlen, T);
    if (T == 0) return DSA_OK;
    const RowSplit rows = row_split_for(selected, idx, T, N, Hq, Hkv, D, K);
    const int ldw = bitmap_ldw(max_seqlen);
    hipStream_t st = (hipStream_t)stream;
    hipError_t e = hipSuccess;
    if (rows.tiles > 0) {
        uint32_t *bitmap = nullptr;
        if (selected) {
            const size_t need = dsa_attn_fwd_workspace_bytes(T, max_seqlen, 1);
            if (!ws || ws_bytes < need) return fail(DSA_ERR_WORKSPACE, "forward workspace: have %zu bytes, need %zu", ws_bytes, need);
            if ((size_t)ldw * 4 > 64 * 1024) return fail(DSA_ERR_UNSUPPORTED, "max_seqlen=%d: selection bitmap row exceeds 64 KiB of LDS", max_seqlen);
            bitmap = (uint32_t *)ws;
            if (build_bitmap) {
                e = dsa_launch_bitmap(idx, n, cu, N, T, K, ldw, bitmap, st);
                if (e != hipSuccess) return hip_fail(e, "bitmap launch");
            }
        }
        const int64_t strides[6] = {(int64_t)Hq * D, D, (int64_t)Hkv * D, D, (int64_t)Hkv * D, D};
        e = dsa_launch_tile_fwd(q, k, v, strides, bitmap, ldw, cu, N, T, Hq, Hkv, D, softmax_scale, rows.tiles, rows.len,
                                rows.below, idx ? 0 : K, dtype == DSA_DTYPE_SPLIT_BF16, causal, out, lse, st);
        if (e != hipSuccess) return hip_fail(e, "tile forward launch");
    }
    if (rows.walks(max_seqlen)) {
        e = dsa_launch_sel_fwd(q, k, v, (const uint32_t *)ws, ldw, cu, N, T, Hq, Hkv, softmax_scale, rows.tiles, rows.walk, rows.len, out, lse, st);
        if (e != hipSuccess) return hip_fail(e, "compacted forward launch");
    }
    if (rows.gathers(max_seqlen, T, N)) {
        e = dsa_launch_attn_fwd(q, k, v, idx, n, cu, N, T, Hq, Hkv, D, K, softmax_scale, rows.walk, rows.len, rows.below, out, lse, st);
        if (e != hipSuccess) return hip_fail(e, "gather forward launch");
    }
    return DSA_OK;
}

extern "C" int dsa_attn_fwd(const void *q, const void *k, const void *v, const int32_t *idx, const int32_t *n,
                            const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale,
                            int dtype, int max_seqlen, int causal, void *out, float *lse, void *ws, size_t ws_bytes,
                            void *stream) {
    return attn_fwd_run(q, k, v, idx != nullptr, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen, causal, out, lse, ws, ws_bytes,
                        1, stream);
}

extern "C" int dsa_attn_fwd_saved_bitmap(const void *q, const void *k, const void *v, const int32_t *idx, const int32_t *n,
                                         const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale,
                                         int dtype, int max_seqlen, int causal, void *out, float *lse, const void *bitmap,
                                         size_t bitmap_bytes, void *stream) {
    if (!idx) return fail(DSA_ERR_ARG, "a saved bitmap belongs to a selection: idx is null");
    return attn_fwd_run(q, k, v, idx != nullptr, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen, causal, out, lse,
                        const_cast<void *>(bitmap), bitmap_bytes, 0, stream);
}

extern "C" int dsa_attn_fwd_words(const void *q, const void *k, const void *v, const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K,
                                  float softmax_scale, int dtype, int max_seqlen, void *out, float *lse, const void *bitmap, size_t bitmap_bytes,
                                  void *stream) {
    return attn_fwd_run(q, k, v, true, nullptr, nullptr, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen, 1, out, lse,
                        const_cast<void *>(bitmap), bitmap_bytes, 0, stream);
}

extern "C" int dsa_index_topk_bitmap(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int T, int N,
                                     int Hi, int Di, int K, float scale, int dtype, int max_seqlen, int32_t *idx, int32_t *n,
                                     float *sel_scores, void *bitmap, size_t bitmap_bytes, void *ws, size_t ws_bytes,
                                     void *stream) {
    if (T > 0 && max_seqlen >= 1) {
        const size_t need = dsa_attn_fwd_workspace_bytes(T, max_seqlen, 1);
        if (!bitmap || bitmap_bytes < need) return fail(DSA_ERR_WORKSPACE, "selection bitmap: have %zu bytes, need %zu", bitmap_bytes, need);
    }
    return index_topk_impl(q_idx, k_idx, w_idx, cu, T, N, Hi, Di, K, scale, dtype, max_seqlen, idx, n, sel_scores,
                           (uint32_t *)bitmap, ws, ws_bytes, stream);
}

extern "C" int dsa_index_topk_words(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *cu, int T, int N, int Hi, int Di, int K,
                                    float scale, int dtype, int max_seqlen, void *bitmap, size_t bitmap_bytes, void *ws, size_t ws_bytes,
                                    void *stream) {
    if (T > 0 && max_seqlen >= 1) {
        const size_t need = dsa_attn_fwd_workspace_bytes(T, max_seqlen, 1);
        if (!bitmap || bitmap_bytes < need) return fail(DSA_ERR_WORKSPACE, "selection bitmap: have %zu bytes, need %zu", bitmap_bytes, need);
    }
    return index_topk_impl(q_idx, k_idx, w_idx, cu, T, N, Hi, Di, K, scale, dtype, max_seqlen, nullptr, nullptr, nullptr, (uint32_t *)bitmap, ws,
                           ws_bytes, stream, true);
}

// ---- attention mass of the selected keys (training target of the indexer) ---------------------------
// bitmap + one (T,K) fp32 table per group of kv heads (none when one group takes all kv heads)
extern "C" size_t dsa_attn_mass_workspace_bytes(int T, int N, int Hq, int Hkv, int D, int K, int max_seqlen) {
    if (T <= 0 || N < 0 || Hkv <= 0 || Hq < Hkv || K <= 0) return 0;
    const int g = dsa_mass_groups(Hq, Hkv, D);
    return align_up((size_t)T * bitmap_ldw(max_seqlen) * 4, 256) + (g > 1 ? align_up((size_t)g * T * K * 4, 256) : 0);
}

// saved_bitmap != NULL: the bitmap of idx/n exists already (left by dsa_index_topk_bitmap or a forward) and is only read;
// ws then holds the partial tables alone
static int attn_mass_run(const void *q, const void *k, const float *lse, const int32_t *idx, const int32_t *n, const int32_t *cu,
                         int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale, int dtype, int max_seqlen, float *mass,
                         const void *saved_bitmap, size_t saved_bytes, void *ws, size_t ws_bytes, void *stream) {
    if (dtype == DSA_DTYPE_SPLIT_BF16) return fail(DSA_ERR_UNSUPPORTED, "q/k/v must be bf16 (dtype code %d)", dtype);
    if (int rc = check_attn(T, N, cu, Hq, Hkv, D, K, dtype, idx != nullptr, idx, n)) return rc;
    if (!q || !k || !lse || !idx || !n || !mass) return fail(DSA_ERR_ARG, "null tensor pointer");
    if (int rc = check_aligned(k, k, "k")) return rc;
    if (max_seqlen < 1 || max_seqlen > (T > 0 ? T : 1)) return fail(DSA_ERR_ARG, "max_seqlen=%d outside [1,T=%d]", max_seqlen, T);
    if (T == 0) return DSA_OK;
    const int ldw = bitmap_ldw(max_seqlen);
    const size_t bm = align_up((size_t)T * ldw * 4, 256);
    const size_t need = dsa_attn_mass_workspace_bytes(T, N, Hq, Hkv, D, K, max_seqlen) - (saved_bitmap ? bm : 0);
    if (need && (!ws || ws_bytes < need)) return fail(DSA_ERR_WORKSPACE, "mass workspace: have %zu bytes, need %zu", ws_bytes, need);
    if (saved_bitmap && saved_bytes < bm) return fail(DSA_ERR_WORKSPACE, "selection bitmap: have %zu bytes, need %zu", saved_bytes, bm);
    if ((size_t)ldw * 4 > 64 * 1024) return fail(DSA_ERR_UNSUPPORTED, "max_seqlen=%d: selection bitmap row exceeds 64 KiB of LDS", max_seqlen);
    hipStream_t st = (hipStream_t)stream;
    const uint32_t *bitmap = saved_bitmap ? (const uint32_t *)saved_bitmap : (const uint32_t *)ws;
    float *partial = (float *)((char *)ws + (saved_bitmap ? 0 : bm));
    hipError_t e = hipSuccess;
    if (!saved_bitmap) {
        e = dsa_launch_bitmap(idx, n, cu, N, T, K, ldw, (uint32_t *)ws, st);
        if (e != hipSuccess) return hip_fail(e, "bitmap launch");
    }
    e = dsa_launch_tile_mass(q, k, lse, bitmap, ldw, n, cu, N, T, Hq, Hkv, D, K, softmax_scale, partial, mass, st);
    if (e != hipSuccess) return hip_fail(e, "attention mass launch");
    return DSA_OK;
}

extern "C" int dsa_attn_mass(const void *q, const void *k, const float *lse, const int32_t *idx, const int32_t *n,
                             const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale,
                             int dtype, int max_seqlen, float *mass, void *ws, size_t ws_bytes, void *stream) {
    return attn_mass_run(q, k, lse, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen, mass, nullptr, 0, ws,
                         ws_bytes, stream);
}

extern "C" int dsa_attn_mass_saved_bitmap(const void *q, const void *k, const float *lse, const int32_t *idx, const int32_t *n,
                                          const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale,
                                          int dtype, int max_seqlen, float *mass, const void *bitmap, size_t bitmap_bytes,
                                          void *ws, size_t ws_bytes, void *stream) {
    if (!bitmap) return fail(DSA_ERR_ARG, "null selection bitmap");
    return attn_mass_run(q, k, lse, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen, mass, bitmap,
                         bitmap_bytes, ws, ws_bytes, stream);
}

// ---- the query-side and the key-side pass of one backward side by side ----
// Both read the same inputs and write different outputs, and a launch of few workgroups ends on its longest walks with
// most CUs idle: the query side then runs on a second stream of the library's own (default priority, one per device,
// made on first use outside any capture) between a fork and a join event, so that to the caller everything still
// happens on the stream it passed.  A stream under capture takes the second one into the capture through the events.
// mode 1 runs the passes side by side for key-side launches of at most this many workgroups (larger ones fill the GPU
// alone) whose work bound T * max_seqlen * Hq * D reaches the second figure: below it the host issues a step more slowly than
// the GPU runs it, and the fork, the join and the pass over dO and O (with the key side's list in the same launch) cost more
// than the overlap gains (head_dim 256 has both passes in one launch instead).  Step times, one after the other -> side by side: head_dim 128 packed
// rows of 4096-8192 tokens, 5-19 % less; 10 000-16 384 tokens, 0-3 % less; 1000 tokens at 2e9, 130 -> 105; 700 tokens at 7e8,
// level.  Without a causal mask the walks of a segment are all equally long, and small launches win nothing.
#define DSA_BWD_OVERLAP_MAX_WG (6 * 256)
#define DSA_ONE_LAUNCH_ROWS 300000                       // (query, head) rows of a launch of both passes, at most (attn_bwd_run)
#define DSA_BWD_OVERLAP_MIN_WORK 2.0e9
#define DSA_BWD_OVERLAP_MIN_WORK_FULL 6.0e10
struct OverlapCtx {
    hipStream_t aux = nullptr;
    hipEvent_t fork = nullptr, join = nullptr;
    bool failed = false;
};
static OverlapCtx g_overlap[DSA_MAX_DEVICES];
static std::mutex g_overlap_mu;                          // held from fork to join: the events are shared by every caller
static std::atomic<int> g_bwd_overlap{1};               // 0 never, 1 launches of few workgroups, 2 always
extern "C" int dsa_set_bwd_overlap(int mode) {
    if (mode < 0 || mode > 2) return fail(DSA_ERR_ARG, "bwd overlap mode=%d outside [0,2]", mode);
    g_bwd_overlap.store(mode, std::memory_order_relaxed);
    return DSA_OK;
}
extern "C" int dsa_get_bwd_overlap(void) { return g_bwd_overlap.load(std::memory_order_relaxed); }
// null when the second stream is not to be had (then the passes run one after the other); call with g_overlap_mu held
static OverlapCtx *overlap_ctx(hipStream_t main_stream) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= DSA_MAX_DEVICES) return nullptr;
    OverlapCtx &c = g_overlap[dev];
    if (c.aux) return &c;
    if (c.failed) return nullptr;
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    if (main_stream && (hipStreamIsCapturing(main_stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone)) {
        (void)hipGetLastError();
        return nullptr;                                  // nothing is created while a capture runs
    }
    if (hipStreamCreateWithFlags(&c.aux, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreateWithFlags(&c.fork, hipEventDisableTiming) != hipSuccess ||
        hipEventCreateWithFlags(&c.join, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        c.aux = nullptr;
        c.failed = true;
        return nullptr;
    }
    return &c;
}

// ---- indexer backward: gradients of the selected scores w.r.t. the indexer's inputs --------------------
extern "C" size_t dsa_indexer_bwd_workspace_bytes(int T, int Di, int max_seqlen) {
    if (T <= 0) return 0;
    const int ldw = bitmap_ldw(max_seqlen);                    // selection bitmap + slot prefix table + partial dk sums + fp32 head weights
    return 2 * align_up((size_t)T * ldw * 4, 256) + align_up(dsa_indexer_bwd_partial_bytes(T, Di, ldw), 256) + (size_t)T * 64 * 4;
}

extern "C" int dsa_indexer_bwd_scaled(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n,
                                      const float *dscore, const float *grad, const int32_t *cu, int T, int N, int Hi, int Di, int K,
                                      float scale, int dtype, int max_seqlen, void *dq_idx, void *dk_idx, void *dw, int dw_dtype, void *ws,
                                      size_t ws_bytes, void *stream) {
    if (int rc = check_packed(T, N, cu)) return rc;
    if (dtype != DSA_DTYPE_BF16) return fail(DSA_ERR_UNSUPPORTED, "indexer tensors must be bf16 (dtype code %d)", dtype);
    if (Hi < 1 || Hi > 64) return fail(DSA_ERR_UNSUPPORTED, "Hi=%d: 1..64 indexer heads", Hi);
    if (!(Di == 64 || Di == 128)) return fail(DSA_ERR_UNSUPPORTED, "Di=%d: the indexer backward covers 64 and 128", Di);
    if (dw_dtype != DSA_DTYPE_BF16 && dw_dtype != DSA_DTYPE_FP32) return fail(DSA_ERR_ARG, "dw dtype code %d", dw_dtype);
    if (K < 1) return fail(DSA_ERR_ARG, "top_k=%d must be >= 1", K);
    if (!q_idx || !k_idx || !w_idx || !idx || !n || !dscore || !dq_idx || !dk_idx || !dw) return fail(DSA_ERR_ARG, "null tensor pointer");
    if (int rc = check_aligned(q_idx, k_idx, "q_idx and k_idx")) return rc;
    if (max_seqlen < 1 || max_seqlen > (T > 0 ? T : 1)) return fail(DSA_ERR_ARG, "max_seqlen=%d outside [1,T=%d]", max_seqlen, T);
    if (T == 0) return DSA_OK;
    const size_t need = dsa_indexer_bwd_workspace_bytes(T, Di, max_seqlen);
    if (!ws || ws_bytes < need) return fail(DSA_ERR_WORKSPACE, "indexer backward workspace: have %zu bytes, need %zu", ws_bytes, need);
    const int ldw = bitmap_ldw(max_seqlen);
    if ((size_t)ldw * 4 > 64 * 1024) return fail(DSA_ERR_UNSUPPORTED, "max_seqlen=%d: selection bitmap row exceeds 64 KiB of LDS", max_seqlen);
    hipStream_t st = (hipStream_t)stream;
    const size_t bm = align_up((size_t)T * ldw * 4, 256);
    uint32_t *bitmap = (uint32_t *)ws;
    int32_t *prefix = (int32_t *)((char *)ws + bm);
    float *partial = (float *)((char *)ws + 2 * bm);
    float *w_f32 = (float *)((char *)ws + need - (size_t)T * 64 * 4);
    hipError_t e = dsa_launch_bitmap(idx, n, cu, N, T, K, ldw, bitmap, st);
    if (e != hipSuccess) return hip_fail(e, "bitmap launch");
    // the query side (dq_idx, dw) and the key side (dk_idx) read the same inputs and write different outputs: side by
    // side on two streams where dsa_set_bwd_overlap allows it, as the two passes of the attention backward
    std::unique_lock<std::mutex> ov_lock;
    OverlapCtx *ov = nullptr;
    const int ov_mode = g_bwd_overlap.load(std::memory_order_relaxed);
    // (mode 1: launches up to 16 384 tokens with T * max_seqlen * Hi * Di of at least 1e10 - 8192 tokens 0.24 -> 0.20 ms,
    // 16 384 tokens 0.53 -> 0.48; at 32 768 tokens both sides fill the GPU alone and nothing is gained)
    if (ov_mode == 2 || (ov_mode == 1 && T <= 16384 && (double)T * max_seqlen * Hi * Di >= 1e10)) {
        ov_lock = std::unique_lock<std::mutex>(g_overlap_mu);
        ov = overlap_ctx(st);
        if (!ov) ov_lock.unlock();
    }
    hipStream_t sq = st;
    if (ov) {
        e = hipEventRecord(ov->fork, st);
        if (e == hipSuccess) e = hipStreamWaitEvent(ov->aux, ov->fork, 0);
        if (e != hipSuccess) return hip_fail(e, "fork to the second stream");
        sq = ov->aux;
    }
    int rc = DSA_OK;
    e = dsa_launch_indexer_bwd(q_idx, k_idx, w_idx, idx, n, dscore, grad, bitmap, prefix, w_f32, ldw, cu, N, T, Hi, Di, K, scale, dq_idx, dk_idx, dw,
                               dw_dtype == DSA_DTYPE_BF16, partial, st, sq);
    if (e != hipSuccess) rc = hip_fail(e, "indexer backward launch");
    if (ov) {
        e = hipEventRecord(ov->join, ov->aux);
        if (e == hipSuccess) e = hipStreamWaitEvent(st, ov->join, 0);
        if (e != hipSuccess && rc == DSA_OK) rc = hip_fail(e, "join of the second stream");
    }
    return rc;
}

extern "C" int dsa_indexer_bwd(const void *q_idx, const void *k_idx, const void *w_idx, const int32_t *idx, const int32_t *n,
                               const float *dscore, const int32_t *cu, int T, int N, int Hi, int Di, int K, float scale,
                               int dtype, int max_seqlen, void *dq_idx, void *dk_idx, float *dw, void *ws, size_t ws_bytes,
                               void *stream) {
    return dsa_indexer_bwd_scaled(q_idx, k_idx, w_idx, idx, n, dscore, nullptr, cu, T, N, Hi, Di, K, scale, dtype, max_seqlen, dq_idx,
                                  dk_idx, dw, DSA_DTYPE_FP32, ws, ws_bytes, stream);
}

extern "C" size_t dsa_attn_bwd_workspace_bytes(int T, int Hq, int max_seqlen, int has_idx) {
    if (T <= 0) return 0;
    size_t b = align_up((size_t)T * Hq * 4, 256);                                     // delta
    if (has_idx) b += align_up((size_t)T * bitmap_ldw(max_seqlen) * 4, 256);          // selection bitmap
    b += align_up(dsa_tile_dkv_partial_bytes(T), 256);                                // dK / dV of key-tile walks in pieces
    return b + align_up(dsa_tile_order_bytes(T), 256);                                // launch order of the key tiles
}

extern "C" size_t dsa_attn_bwd_bitmap_offset(int T, int Hq) {
    if (T <= 0 || Hq <= 0) return 0;
    return align_up((size_t)T * Hq * 4, 256);
}

// the backward proper: every buffer named, so that the two entry points below differ only in where the buffers live
static int attn_bwd_run(const void *dout, const void *q, const void *k, const void *v, const void *out, const float *lse,
                        bool selected, const int32_t *idx, const int32_t *n, const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K,
                        float softmax_scale, int max_seqlen, int causal, void *dq, void *dk, void *dv, float *delta,
                        uint32_t *bitmap, float *partial, size_t partial_bytes, int32_t *order, int parts, hipStream_t st,
                        bool carried = false) {
    const int ldw = bitmap_ldw(max_seqlen);
    if (selected && (size_t)ldw * 4 > 64 * 1024) return fail(DSA_ERR_UNSUPPORTED, "max_seqlen=%d: selection bitmap row exceeds 64 KiB of LDS", max_seqlen);
    const RowSplit rows = row_split_for(selected, idx, T, N, Hq, Hkv, D, K);
    hipError_t e = hipSuccess;
    // the two passes side by side on two streams: launches of few workgroups only (larger ones fill the GPU alone)
    std::unique_lock<std::mutex> ov_lock;
    OverlapCtx *ov = nullptr;
    const int ov_mode = g_bwd_overlap.load(std::memory_order_relaxed);
    // head_dim 256: both passes in one launch (dsa_tile_bwd.hip), or, where that does not pay, one after the other.  It saves a launch and the idle CUs of
    // the key side's end; the pass over dO and O that dQ has inside it when it runs first comes back, and that grows with the rows.  Backward, us, one
    // after the other -> one launch, 16 heads over 2: 300 tokens 73 -> 54, 2500 253 -> 190, eight segments of 512 137 -> 118, 16 of 1000 562 -> 537, 4 of 4000 2009 ->
    // 1593, 4 of 8000 (512 000 rows) 5852 -> 5852, 48 of 1000 (768 000) 1590 -> 1616; 16 over 4: 16 000 tokens 5718 -> 5682, 4 of 8000 with a selection 5712 -> 5872;
    // 8 over 8: 4 of 4000 814 -> 804, 48 of 1000 (384 000) 1013 -> 1042; 32 over 8: 4 of 4000 (512 000) 3108 -> 3182, 4 of 8000 11 560 -> 11 813; fp32 rows of 64, 16 over 8: 4 of
    // 4000 1197 -> 1194, 4 of 8000 4399 -> 4553, 48 of 1000 1502 -> 1558.  200 segments of 100 (640 000) 743 -> 674: of short ones whatever the rows.
    const bool both = (parts & DSA_BWD_DQ) && (parts & DSA_BWD_DKV) && ov_mode > 0;
    const bool may_share = both && D == 256 && max_seqlen <= rows.below && !(((uintptr_t)q | (uintptr_t)dout) & 15);
    const bool one_launch = may_share && (ov_mode == 2 || (int64_t)T * Hq <= DSA_ONE_LAUNCH_ROWS || T / 256 <= N);
    if (both && !may_share) {
        const int64_t dkv_wg = ((int64_t)T / 128 + N) * Hkv * (D > 128 ? 2 : 1);     // (head_dim 256: one workgroup per CU, half as many fill it)
        const double work = (double)T * max_seqlen * Hq * D;
        if (ov_mode == 2 || (dkv_wg <= DSA_BWD_OVERLAP_MAX_WG && work >= (causal ? DSA_BWD_OVERLAP_MIN_WORK : DSA_BWD_OVERLAP_MIN_WORK_FULL))) {
            ov_lock = std::unique_lock<std::mutex>(g_overlap_mu);
            ov = overlap_ctx(st);
            if (!ov) ov_lock.unlock();
        }
    }
    // delta = rowsum(dO * O): a pass of its own, unless the tile dQ kernel of the same call owns every query row
    // (no row beyond the tile/gather split) - then that kernel forms it from the dO rows it loads anyway - and the
    // key side, which reads every delta, runs after it
    const bool fuse_delta = (parts & DSA_BWD_DELTA) && (parts & DSA_BWD_DQ) && rows.tiles > 0 && !rows.walks(max_seqlen) && !rows.gathers(max_seqlen, T, N) && !ov && !one_launch;
    int listed = 0;                                      // the launch order of the key tiles is there
    if ((parts & DSA_BWD_DELTA) && (ov || one_launch)) {
        e = dsa_launch_tile_order_delta(dout, out, cu, N, T, Hq, Hkv, D, selected, causal, order, partial, partial_bytes, delta, st);
        if (e == hipSuccess) listed = 1;
        else if (e != hipErrorNotReady) return hip_fail(e, "order and delta launch");   // (not ready: this launch needs no list)
    }
    if ((parts & DSA_BWD_DELTA) && !fuse_delta && !listed) {
        e = dsa_launch_delta(dout, out, T, Hq, D, delta, st);
        if (e != hipSuccess) return hip_fail(e, "delta launch");
    }
    if ((parts & DSA_BWD_BITMAP) && idx) {
        e = dsa_launch_bitmap(idx, n, cu, N, T, K, ldw, bitmap, st);
        if (e != hipSuccess) return hip_fail(e, "bitmap launch");
    }
    hipStream_t sq = st;
    if (ov) {
        e = hipEventRecord(ov->fork, st);
        if (e == hipSuccess) e = hipStreamWaitEvent(ov->aux, ov->fork, 0);
        if (e != hipSuccess) return hip_fail(e, "fork to the second stream");
        sq = ov->aux;
    }
    int rc = DSA_OK;
    const int walk_len = key_walk_len(selected, q, dout, T, N, Hq, Hkv, D, K);
    const DqBeside beside{idx ? 0 : K, dq};
    auto key_side = [&]() {
        hipError_t e = dsa_launch_tile_dkv(dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, D, softmax_scale, carried, causal, walk_len, order, listed,
                                           partial, partial_bytes, dk, dv, one_launch ? &beside : nullptr, st);
        if (e == hipSuccess && max_seqlen >= walk_len)
            e = dsa_launch_selkv(dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, softmax_scale, walk_len, dk, dv, st);
        return e == hipSuccess ? DSA_OK : hip_fail(e, "dkv launch");
    };
    // (side by side, the key side is issued first: it is the longer pass and starts with its longest walks)
    if (ov) rc = key_side();
    if (rc == DSA_OK && (parts & DSA_BWD_DQ) && !one_launch) {
        if (rows.tiles > 0) {
            e = dsa_launch_tile_dq(dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, D, softmax_scale, rows.tiles, rows.len,
                                   rows.below, idx ? 0 : K, carried, causal, dq, fuse_delta ? out : nullptr, delta, sq);
            if (e != hipSuccess) rc = hip_fail(e, "tile dq launch");
        }
        if (rc == DSA_OK && rows.walks(max_seqlen)) {
            e = dsa_launch_sel_dq(dout, q, k, v, lse, delta, bitmap, ldw, cu, N, T, Hq, Hkv, softmax_scale, rows.tiles, rows.walk, rows.len, dq, sq);
            if (e != hipSuccess) rc = hip_fail(e, "compacted dq launch");
        }
        if (rc == DSA_OK && rows.gathers(max_seqlen, T, N)) {
            e = dsa_launch_gather_dq(dout, q, k, v, lse, delta, idx, n, cu, N, T, Hq, Hkv, D, K, softmax_scale, rows.walk, rows.len, rows.below, dq, sq);
            if (e != hipSuccess) rc = hip_fail(e, "gather dq launch");
        }
    }
    if (rc == DSA_OK && !ov && (parts & DSA_BWD_DKV)) rc = key_side();
    if (ov) {                                            // joined also after a failed launch: the caller's stream stays whole
        e = hipEventRecord(ov->join, ov->aux);
        if (e == hipSuccess) e = hipStreamWaitEvent(st, ov->join, 0);
        if (e != hipSuccess && rc == DSA_OK) rc = hip_fail(e, "join of the second stream");
    }
    return rc;
}

static int check_bwd(const void *dout, const void *q, const void *k, const void *v, const void *out, const float *lse,
                     bool selected, const int32_t *idx, const int32_t *n, const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K,
                     int dtype, int max_seqlen, int causal, const void *dq, const void *dk, const void *dv) {
    if (int rc = check_attn(T, N, cu, Hq, Hkv, D, K, dtype, selected, idx, n)) return rc;
    if (!causal && selected) return fail(DSA_ERR_ARG, "a key selection (idx) implies causal attention");
    if (!dout || !q || !k || !v || !out || !lse || !dq || !dk || !dv) return fail(DSA_ERR_ARG, "null tensor pointer");
    if (int rc = check_aligned(k, v, "k and v")) return rc;
    if (max_seqlen < 1 || max_seqlen > (T > 0 ? T : 1)) return fail(DSA_ERR_ARG, "max_seqlen=%d outside [1,T=%d]", max_seqlen, T);
    return DSA_OK;
}

extern "C" int dsa_attn_bwd_parts(const void *dout, const void *q, const void *k, const void *v, const void *out,
                                  const float *lse, const int32_t *idx, const int32_t *n, const int32_t *cu, int T,
                                  int N, int Hq, int Hkv, int D, int K, float softmax_scale, int dtype, int max_seqlen,
                                  int causal, void *dq, void *dk, void *dv, void *ws, size_t ws_bytes, int parts,
                                  void *stream) {
    if (int rc = check_bwd(dout, q, k, v, out, lse, idx != nullptr, idx, n, cu, T, N, Hq, Hkv, D, K, dtype, max_seqlen, causal, dq, dk, dv)) return rc;
    if (T == 0) return DSA_OK;
    const size_t need = dsa_attn_bwd_workspace_bytes(T, Hq, max_seqlen, idx != nullptr);
    if (!ws || ws_bytes < need) return fail(DSA_ERR_WORKSPACE, "backward workspace: have %zu bytes, need %zu", ws_bytes, need);
    float *delta = (float *)ws;
    uint32_t *bitmap = idx ? (uint32_t *)((char *)ws + dsa_attn_bwd_bitmap_offset(T, Hq)) : nullptr;
    int32_t *order = (int32_t *)((char *)ws + need - align_up(dsa_tile_order_bytes(T), 256));
    const size_t partial_bytes = dsa_tile_dkv_partial_bytes(T);
    float *partial = partial_bytes ? (float *)((char *)order - align_up(partial_bytes, 256)) : nullptr;
    return attn_bwd_run(dout, q, k, v, out, lse, idx != nullptr, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, max_seqlen, causal, dq, dk, dv,
                        delta, bitmap, partial, partial_bytes, order, parts, (hipStream_t)stream, dtype == DSA_DTYPE_SPLIT_BF16);
}

// Scratch of the backward that nothing outlives: delta, the launch order of the key tiles and - only for launches small
// enough to be cut into pieces (dkv_pieces_max_wg workgroups before the cut) - the fp32 partial sums of those pieces.
static size_t bwd_partial_bytes_for(int T, int N, int Hkv, int D) {
    if (((int64_t)T / 128 + N) * Hkv > dkv_pieces_max_wg(D)) return 0;
    return dsa_tile_dkv_partial_bytes(T);
}
extern "C" size_t dsa_attn_bwd_scratch_bytes(int T, int N, int Hq, int Hkv, int D) {
    if (T <= 0 || N < 0 || Hq <= 0 || Hkv <= 0) return 0;
    return align_up((size_t)T * Hq * 4, 256) + align_up(bwd_partial_bytes_for(T, N, Hkv, D), 256) +
           align_up(dsa_tile_order_bytes(T), 256);
}

static int attn_bwd_saved(const void *dout, const void *q, const void *k, const void *v, const void *out, const float *lse, bool selected,
                          const int32_t *idx, const int32_t *n, const int32_t *cu, int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale,
                          int dtype, int max_seqlen, int causal, void *dq, void *dk, void *dv, const void *fwd_ws, size_t fwd_ws_bytes, void *scratch,
                          size_t scratch_bytes, void *stream) {
    if (int rc = check_bwd(dout, q, k, v, out, lse, selected, idx, n, cu, T, N, Hq, Hkv, D, K, dtype, max_seqlen, causal, dq, dk, dv)) return rc;
    if (T == 0) return DSA_OK;
    if (selected) {
        if (row_split_for(selected, idx, T, N, Hq, Hkv, D, K).tiles <= 0) return fail(DSA_ERR_ARG, "with the tile crossover at 0 the forward builds no bitmap: use dsa_attn_bwd");
        const size_t have = dsa_attn_fwd_workspace_bytes(T, max_seqlen, 1);
        if (!fwd_ws || fwd_ws_bytes < have) return fail(DSA_ERR_WORKSPACE, "forward workspace (selection bitmap): have %zu bytes, need %zu", fwd_ws_bytes, have);
    }
    const size_t need = dsa_attn_bwd_scratch_bytes(T, N, Hq, Hkv, D);
    if (!scratch || scratch_bytes < need) return fail(DSA_ERR_WORKSPACE, "backward scratch: have %zu bytes, need %zu", scratch_bytes, need);
    float *delta = (float *)scratch;
    const size_t partial_bytes = bwd_partial_bytes_for(T, N, Hkv, D);
    float *partial = partial_bytes ? (float *)((char *)scratch + align_up((size_t)T * Hq * 4, 256)) : nullptr;
    int32_t *order = (int32_t *)((char *)scratch + need - align_up(dsa_tile_order_bytes(T), 256));
    // the kernels only read the bitmap; the forward's workspace is not written here
    uint32_t *bitmap = selected ? const_cast<uint32_t *>((const uint32_t *)fwd_ws) : nullptr;
    return attn_bwd_run(dout, q, k, v, out, lse, selected, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, max_seqlen, causal, dq, dk, dv,
                        delta, bitmap, partial, partial_bytes, order, DSA_BWD_ALL & ~DSA_BWD_BITMAP, (hipStream_t)stream,
                        dtype == DSA_DTYPE_SPLIT_BF16);
}

extern "C" int dsa_attn_bwd_saved_bitmap(const void *dout, const void *q, const void *k, const void *v, const void *out,
                                         const float *lse, const int32_t *idx, const int32_t *n, const int32_t *cu, int T,
                                         int N, int Hq, int Hkv, int D, int K, float softmax_scale, int dtype,
                                         int max_seqlen, int causal, void *dq, void *dk, void *dv, const void *fwd_ws,
                                         size_t fwd_ws_bytes, void *scratch, size_t scratch_bytes, void *stream) {
    return attn_bwd_saved(dout, q, k, v, out, lse, idx != nullptr, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen, causal, dq, dk, dv,
                          fwd_ws, fwd_ws_bytes, scratch, scratch_bytes, stream);
}

extern "C" int dsa_attn_bwd_words(const void *dout, const void *q, const void *k, const void *v, const void *out, const float *lse, const int32_t *cu,
                                  int T, int N, int Hq, int Hkv, int D, int K, float softmax_scale, int dtype, int max_seqlen, void *dq, void *dk,
                                  void *dv, const void *bitmap, size_t bitmap_bytes, void *scratch, size_t scratch_bytes, void *stream) {
    return attn_bwd_saved(dout, q, k, v, out, lse, true, nullptr, nullptr, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen, 1, dq, dk, dv,
                          bitmap, bitmap_bytes, scratch, scratch_bytes, stream);
}

extern "C" int dsa_dense_bwd_rows(const void *dout, const void *q, const void *k, const void *v, const void *out, const float *lse,
                                  const int32_t *cu, int T, int N, int Hq, int Hkv, int D, float softmax_scale, int dtype,
                                  int max_seqlen, int causal, void *dq, void *dk, void *dv, void *scratch, size_t scratch_bytes,
                                  void *stream) {
    if (D < 8 || D > 128 || D % 8) return fail(DSA_ERR_UNSUPPORTED, "head_dim=%d: need a multiple of 8 up to 128", D);
    if (int rc = check_bwd(dout, q, k, v, out, lse, false, nullptr, nullptr, cu, T, N, Hq, Hkv, 64, 0, dtype, max_seqlen, causal, dq, dk, dv)) return rc;
    if (T == 0) return DSA_OK;
    const size_t need = dsa_attn_bwd_scratch_bytes(T, N, Hq, Hkv, D);
    if (!scratch || scratch_bytes < need) return fail(DSA_ERR_WORKSPACE, "backward scratch: have %zu bytes, need %zu", scratch_bytes, need);
    const size_t partial_bytes = bwd_partial_bytes_for(T, N, Hkv, D);
    float *partial = partial_bytes ? (float *)((char *)scratch + align_up((size_t)T * Hq * 4, 256)) : nullptr;
    int32_t *order = (int32_t *)((char *)scratch + need - align_up(dsa_tile_order_bytes(T), 256));
    return attn_bwd_run(dout, q, k, v, out, lse, false, nullptr, nullptr, cu, T, N, Hq, Hkv, D, 0, softmax_scale, max_seqlen, causal, dq, dk, dv,
                        (float *)scratch, nullptr, partial, partial_bytes, order, DSA_BWD_ALL & ~DSA_BWD_BITMAP, (hipStream_t)stream);
}

extern "C" int dsa_attn_bwd(const void *dout, const void *q, const void *k, const void *v, const void *out,
                            const float *lse, const int32_t *idx, const int32_t *n, const int32_t *cu, int T, int N,
                            int Hq, int Hkv, int D, int K, float softmax_scale, int dtype, int max_seqlen, int causal,
                            void *dq, void *dk, void *dv, void *ws, size_t ws_bytes, void *stream) {
    return dsa_attn_bwd_parts(dout, q, k, v, out, lse, idx, n, cu, T, N, Hq, Hkv, D, K, softmax_scale, dtype, max_seqlen,
                              causal, dq, dk, dv, ws, ws_bytes, DSA_BWD_ALL, stream);
}

extern "C" int dsa_dense_fwd(const void *q, const void *k, const void *v, const int32_t *cu, int T, int N, int Hq, int Hkv,
                             int D, float softmax_scale, int dtype, int max_seqlen, int causal, void *out, float *lse,
                             void *stream) {
    return dsa_attn_fwd(q, k, v, nullptr, nullptr, cu, T, N, Hq, Hkv, D, 0, softmax_scale, dtype, max_seqlen, causal, out, lse,
                        nullptr, 0, stream);
}

extern "C" int dsa_dense_fwd_strided(const void *q, int64_t q_tok, int64_t q_head, const void *k, int64_t k_tok, int64_t k_head, const void *v,
                                     int64_t v_tok, int64_t v_head, const int32_t *cu, int T, int N, int Hq, int Hkv, int D,
                                     float softmax_scale, int dtype, int max_seqlen, int causal, void *out, float *lse, void *stream) {
    if (D < 8 || D > 256 || D % 8) return fail(DSA_ERR_UNSUPPORTED, "head_dim=%d: need a multiple of 8 up to 256", D);
    if (int rc = check_attn(T, N, cu, Hq, Hkv, 64, 0, dtype, false, nullptr, nullptr)) return rc;     // (head_dim checked above)
    if (!q || !k || !v || !out || !lse) return fail(DSA_ERR_ARG, "null tensor pointer");
    if (max_seqlen < 1 || max_seqlen > (T > 0 ? T : 1)) return fail(DSA_ERR_ARG, "max_seqlen=%d outside [1,T=%d]", max_seqlen, T);
    const int64_t strides[6] = {q_tok, q_head, k_tok, k_head, v_tok, v_head};
    for (int i = 0; i < 6; ++i)
        if (strides[i] < 0 || strides[i] % 8 || (i % 2 == 0 && strides[i] >= (1 << 24)))
            return fail(DSA_ERR_ARG, "strides must be multiples of 8, token strides below 2^24");
    if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15) return fail(DSA_ERR_ARG, "tensors must lie on 16-byte boundaries");
    if (T == 0) return DSA_OK;
    const hipError_t e = dsa_launch_tile_fwd(q, k, v, strides, nullptr, 0, cu, N, T, Hq, Hkv, D, softmax_scale, INT32_MAX, 0, INT32_MAX, 0, 0, causal, out, lse,
                                             (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "tile forward launch");
}

extern "C" int dsa_dense_bwd(const void *dout, const void *q, const void *k, const void *v, const void *out, const float *lse,
                             const int32_t *cu, int T, int N, int Hq, int Hkv, int D, float softmax_scale, int dtype,
                             int max_seqlen, int causal, void *dq, void *dk, void *dv, void *ws, size_t ws_bytes,
                             void *stream) {
    return dsa_attn_bwd(dout, q, k, v, out, lse, nullptr, nullptr, cu, T, N, Hq, Hkv, D, 0, softmax_scale, dtype, max_seqlen,
                        causal, dq, dk, dv, ws, ws_bytes, stream);
}

// ---------------------------------------------------------------------------------------------------
// prologue / gate
// ---------------------------------------------------------------------------------------------------
static int check_prologue(int T, int Hq, int Hkv, int D, int R, int cs_dtype, int64_t q_head, int64_t k_head) {
    if (T < 0 || Hq < 1 || Hkv < 1) return fail(DSA_ERR_ARG, "T=%d Hq=%d Hkv=%d", T, Hq, Hkv);
    if (!(D == 64 || D == 128 || D == 256)) return fail(DSA_ERR_UNSUPPORTED, "head_dim=%d: need 64, 128 or 256", D);
    if (R < 0 || R > D || R % 16) return fail(DSA_ERR_UNSUPPORTED, "rotary width R=%d: need a multiple of 16 up to head_dim=%d", R, D);
    if (cs_dtype != DSA_DTYPE_BF16 && cs_dtype != DSA_DTYPE_FP32) return fail(DSA_ERR_ARG, "cos/sin dtype code %d", cs_dtype);
    if (q_head % 8 || k_head % 8) return fail(DSA_ERR_ARG, "head strides must be multiples of 8 elements (16-byte rows)");
    return DSA_OK;
}

extern "C" size_t dsa_qk_norm_rope_bwd_workspace_bytes(int T, int D) {
    if (T <= 0 || D <= 0) return 0;
    return (size_t)dsa_prologue_bwd_blocks(T) * 2 * D * sizeof(float);
}

extern "C" int dsa_qk_norm_rope_fwd(const void *q_in, int64_t q_tok, int64_t q_head, const void *k_in, int64_t k_tok,
                                    int64_t k_head, const void *qw, const void *kw, float eps, int norm_flags,
                                    const void *cosp, const void *sinp, int cs_dtype, int R, int T, int Hq, int Hkv, int D,
                                    void *q_out, void *k_out, float *q_rstd, float *k_rstd, void *stream) {
    if (int rc = check_prologue(T, Hq, Hkv, D, R, cs_dtype, q_head, k_head)) return rc;
    if (!q_in || !k_in || !qw || !kw || !q_out || !k_out || !q_rstd || !k_rstd || (R > 0 && (!cosp || !sinp)))
        return fail(DSA_ERR_ARG, "null tensor pointer");
    if (q_tok % 8 || k_tok % 8) return fail(DSA_ERR_ARG, "token strides must be multiples of 8 elements");
    hipError_t e = dsa_launch_qk_norm_rope_fwd(q_in, q_tok, q_head, k_in, k_tok, k_head, qw, kw, (norm_flags & DSA_NORM_WEIGHT_BF16) != 0, eps,
                                               (norm_flags & DSA_NORM_OFFSET) ? 1.f : 0.f,
                                               cosp, sinp, cs_dtype == DSA_DTYPE_FP32, R, T, Hq, Hkv, D, q_out, k_out, q_rstd,
                                               k_rstd, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "qk_norm_rope forward launch");
}

extern "C" int dsa_qk_norm_rope_bwd(const void *gq, const void *gk, const void *q_in, int64_t q_tok, int64_t q_head,
                                    const void *k_in, int64_t k_tok, int64_t k_head, const void *qw, const void *kw,
                                    int norm_flags, const void *cosp, const void *sinp, int cs_dtype, int R,
                                    const float *q_rstd, const float *k_rstd, int T, int Hq, int Hkv, int D, void *dq_in,
                                    int64_t dq_tok, int64_t dq_head, void *dk_in, int64_t dk_tok, int64_t dk_head,
                                    float *dqw, float *dkw, void *ws, size_t ws_bytes, void *stream) {
    if (int rc = check_prologue(T, Hq, Hkv, D, R, cs_dtype, q_head, k_head)) return rc;
    if (!gq || !gk || !q_in || !k_in || !qw || !kw || !q_rstd || !k_rstd || !dq_in || !dk_in || !dqw || !dkw ||
        (R > 0 && (!cosp || !sinp)))
        return fail(DSA_ERR_ARG, "null tensor pointer");
    if (q_tok % 8 || k_tok % 8 || dq_tok % 8 || dk_tok % 8 || dq_head % 8 || dk_head % 8)
        return fail(DSA_ERR_ARG, "strides must be multiples of 8 elements");
    const size_t need = dsa_qk_norm_rope_bwd_workspace_bytes(T, D);
    if (need && (!ws || ws_bytes < need)) return fail(DSA_ERR_WORKSPACE, "prologue backward workspace: have %zu bytes, need %zu", ws_bytes, need);
    hipError_t e = dsa_launch_qk_norm_rope_bwd(gq, gk, q_in, q_tok, q_head, k_in, k_tok, k_head, qw, kw, (norm_flags & DSA_NORM_WEIGHT_BF16) != 0,
                                               (norm_flags & DSA_NORM_OFFSET) ? 1.f : 0.f,
                                               cosp, sinp, cs_dtype == DSA_DTYPE_FP32, R, q_rstd, k_rstd, T, Hq, Hkv, D, dq_in,
                                               dq_tok, dq_head, dk_in, dk_tok, dk_head, dqw, dkw, (norm_flags & DSA_NORM_GRAD_BF16) != 0, (float *)ws,
                                               (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "qk_norm_rope backward launch");
}

extern "C" int dsa_sigmoid_gate_fwd(const void *x, const void *gate, int64_t gate_tok, int64_t gate_head, int T, int H, int D,
                                    void *y, void *stream) {
    if (T < 0 || H < 1 || D < 8 || D % 8 || gate_tok % 8 || gate_head % 8) return fail(DSA_ERR_ARG, "T=%d H=%d D=%d or strides not multiples of 8", T, H, D);
    if (!x || !gate || !y) return fail(DSA_ERR_ARG, "null tensor pointer");
    hipError_t e = dsa_launch_sigmoid_gate_fwd(x, gate, gate_tok, gate_head, D, H, T, y, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "sigmoid gate forward launch");
}

extern "C" int dsa_sigmoid_gate_bwd(const void *gy, const void *x, const void *gate, int64_t gate_tok, int64_t gate_head,
                                    int T, int H, int D, void *dx, void *dgate, int64_t dgate_tok, int64_t dgate_head,
                                    void *stream) {
    if (T < 0 || H < 1 || D < 8 || D % 8 || gate_tok % 8 || gate_head % 8 || dgate_tok % 8 || dgate_head % 8)
        return fail(DSA_ERR_ARG, "T=%d H=%d D=%d or strides not multiples of 8", T, H, D);
    if (!gy || !x || !gate || !dx || !dgate) return fail(DSA_ERR_ARG, "null tensor pointer");
    hipError_t e = dsa_launch_sigmoid_gate_bwd(gy, x, gate, gate_tok, gate_head, D, H, T, dx, dgate, dgate_tok, dgate_head,
                                               (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "sigmoid gate backward launch");
}

// ---- several (T, width) bf16 tensors side by side in one row-major buffer ----
extern "C" int dsa_pack_columns(int n, const void *const *src, const int32_t *width, const int32_t *group, const int32_t *dst_col,
                                const int32_t *dst_group, int T, void *dst, int64_t dst_row, void *stream) {
    if (n < 1 || n > DSA_PACK_MAX || T < 0 || !src || !width || !group || !dst_col || !dst_group || dst_row < 8 || dst_row % 8)
        return fail(DSA_ERR_ARG, "n=%d T=%d row=%lld", n, T, (long long)dst_row);
    for (int i = 0; i < n; ++i) {
        if (width[i] < 8 || width[i] % 8 || group[i] < 8 || group[i] % 8 || width[i] % group[i] || dst_col[i] < 0 || dst_col[i] % 8 ||
            dst_group[i] < group[i] || dst_group[i] % 8 || dst_col[i] + (int64_t)(width[i] / group[i] - 1) * dst_group[i] + group[i] > dst_row)
            return fail(DSA_ERR_ARG, "source %d: width %d in groups of %d at column %d, %d apart", i, width[i], group[i], dst_col[i], dst_group[i]);
        if (T > 0 && (!src[i] || ((uintptr_t)src[i] & 15))) return fail(DSA_ERR_ARG, "source %d: null or not on a 16-byte boundary", i);
    }
    if (T == 0) return DSA_OK;
    if (!dst || ((uintptr_t)dst & 15)) return fail(DSA_ERR_ARG, "destination null or not on a 16-byte boundary");
    hipError_t e = dsa_launch_pack_columns(n, src, width, group, dst_col, dst_group, T, dst, dst_row, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "pack columns launch");
}

// ---- fp32 operands carried as stacked split-bf16 rows (the host operator's fp32 path for head_dim <= 64) ----
extern "C" int dsa_split_bf16_stack(const float *x, int64_t rows, int D, int order, void *y, void *stream) {
    if (rows < 0 || D < 4 || D % 4 || (order != 0 && order != 1)) return fail(DSA_ERR_ARG, "rows=%lld D=%d order=%d", (long long)rows, D, order);
    if (rows > 0 && (!x || !y)) return fail(DSA_ERR_ARG, "null tensor pointer");
    hipError_t e = dsa_launch_split_stack(x, rows, D, order, y, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "split/stack launch");
}
extern "C" int dsa_split_bf16_combine(const void *y, int64_t rows, int D, int part, float *out, void *stream) {
    if (rows < 0 || D < 4 || D % 4 || part < 1 || part > 3) return fail(DSA_ERR_ARG, "rows=%lld D=%d part=%d", (long long)rows, D, part);
    if (rows > 0 && (!y || !out)) return fail(DSA_ERR_ARG, "null tensor pointer");
    hipError_t e = dsa_launch_split_combine(y, rows, D, part, out, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "split/combine launch");
}
extern "C" int dsa_split_bf16_stack_qkv(const float *q, const float *k, const float *v, int64_t rows_q, int64_t rows_kv, int D,
                                        void *yq, void *yk, void *yv, void *stream) {
    if (rows_q < 0 || rows_kv < 0 || D < 4 || D % 4) return fail(DSA_ERR_ARG, "rows_q=%lld rows_kv=%lld D=%d", (long long)rows_q, (long long)rows_kv, D);
    if ((rows_q > 0 && (!q || !yq)) || (rows_kv > 0 && (!k || !v || !yk || !yv))) return fail(DSA_ERR_ARG, "null tensor pointer");
    hipError_t e = dsa_launch_split_stack_qkv(q, k, v, rows_q, rows_kv, D, yq, yk, yv, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "split/stack launch");
}
extern "C" int dsa_split_bf16_combine_qkv(const void *yq, const void *yk, const void *yv, int64_t rows_q, int64_t rows_kv, int D,
                                          float *dq, float *dk, float *dv, void *stream) {
    if (rows_q < 0 || rows_kv < 0 || D < 4 || D % 4) return fail(DSA_ERR_ARG, "rows_q=%lld rows_kv=%lld D=%d", (long long)rows_q, (long long)rows_kv, D);
    if ((rows_q > 0 && (!yq || !dq)) || (rows_kv > 0 && (!yk || !yv || !dk || !dv))) return fail(DSA_ERR_ARG, "null tensor pointer");
    hipError_t e = dsa_launch_split_combine_qkv(yq, yk, yv, rows_q, rows_kv, D, dq, dk, dv, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "split/combine launch");
}

// ---- three fp32 arrays rounded to bf16 by one launch (the indexer's inputs of an fp32 caller) ----
extern "C" int dsa_round_bf16_x3(const float *a, const float *b, const float *c, int64_t na, int64_t nb, int64_t nc, void *ya,
                                 void *yb, void *yc, void *stream) {
    if (na < 0 || nb < 0 || nc < 0) return fail(DSA_ERR_ARG, "negative element count");
    if ((na > 0 && (!a || !ya)) || (nb > 0 && (!b || !yb)) || (nc > 0 && (!c || !yc))) return fail(DSA_ERR_ARG, "null tensor pointer");
    if ((((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) || (((uintptr_t)ya | (uintptr_t)yb | (uintptr_t)yc) & 7))
        return fail(DSA_ERR_ARG, "inputs must be 16-byte aligned, outputs 8-byte aligned");
    hipError_t e = dsa_launch_round_bf16_x3(a, b, c, na, nb, nc, ya, yb, yc, (hipStream_t)stream);
    return e == hipSuccess ? DSA_OK : hip_fail(e, "bf16 rounding launch");
}
