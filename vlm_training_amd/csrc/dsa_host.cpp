// Host side of the operators in C++: argument checks, allocations, the C-ABI calls and the autograd nodes, bound to
// Python as vlm_training_amd._dsa_host.
//
// A step of the operator is seven to twelve launches.  Driven from Python (ctypes calls, torch.empty, a Python autograd
// node whose backward takes the interpreter lock) it took the host 110-190 us to issue one, as long as the GPU needs for
// 2048 tokens; the nodes below issue the same calls without the interpreter.  Everything here is ordered on torch's
// current stream of the tensors' device; the arithmetic is in the kernels behind include/dsa_attn.h.
#include <torch/extension.h>

#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <optional>
#include <vector>

#include "../../include/dsa_attn.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

void check(int rc, const char *what) {
    if (rc == 0) return;
    const std::string msg = std::string(what) + " failed (" + std::to_string(rc) + "): " + dsa_last_error();
    if (rc == DSA_ERR_ARG) TORCH_CHECK_VALUE(false, msg);
    TORCH_CHECK(false, msg);
}

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
const int32_t *iptr(const Tensor &t) { return t.defined() ? t.data_ptr<int32_t>() : nullptr; }
float *fptr(const Tensor &t) { return t.defined() ? t.data_ptr<float>() : nullptr; }
void *stream_of(const Tensor &t) { return (void *)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }

void need_gpu(const Tensor &t) {
    if (t.defined() && !t.is_cuda())
        TORCH_CHECK(false, "dsa attention runs on the GPU only (tensor on ", t.device().str(), "); there is no CPU path");
}

// The operators have no forward-mode derivative.  Asked of every differentiable input before anything else: a dual tensor need not
// require a gradient, so a call that builds no graph would drop its tangent without a word.
bool has_tangent(const Tensor &t) { return t.defined() && t._fw_grad(0).defined(); }
void no_forward_mode(std::initializer_list<const Tensor *> inputs, const char *what) {
    for (const Tensor *t : inputs)
        TORCH_CHECK_NOT_IMPLEMENTED(!has_tangent(*t), what, ": forward-mode differentiation is not implemented");
}

Tensor empty(at::IntArrayRef size, at::ScalarType dtype, const Tensor &like) {
    return Tensor(at::detail::empty_cuda(size, dtype, like.device(), std::nullopt));
}
Tensor empty_bytes(size_t bytes, const Tensor &like) { return empty({(int64_t)std::max<size_t>(bytes, 4)}, at::kByte, like); }

bool aligned16(const Tensor &t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }
// contiguous bf16 on a 16-byte boundary: keys, values and index queries go into LDS 16 bytes at a time (a view can start anywhere)
Tensor as_bf16(const Tensor &t) {
    const Tensor c = (t.scalar_type() == at::kBFloat16 ? t : t.to(at::kBFloat16)).contiguous();
    return aligned16(c) ? c : c.clone();
}

Tensor checked_cu(const Tensor &cu) {
    TORCH_CHECK_VALUE(cu.dim() == 1 && cu.numel() >= 2, "cu_seqlens must be 1-D with at least two entries");
    return (cu.scalar_type() == at::kInt ? cu : cu.to(at::kInt)).contiguous();
}

// the indexer's three inputs in bf16; three fp32 ones by one launch, into one buffer with every part on a 16-byte boundary
struct IndexInputs { Tensor q, k, w; };
IndexInputs index_inputs(const Tensor &a_, const Tensor &b_, const Tensor &c_) {
    if (!(a_.scalar_type() == at::kFloat && b_.scalar_type() == at::kFloat && c_.scalar_type() == at::kFloat && a_.numel()))
        return {as_bf16(a_), as_bf16(b_), as_bf16(c_)};
    const Tensor a = a_.contiguous(), b = b_.contiguous(), c = c_.contiguous();
    if (((uintptr_t)a.data_ptr() | (uintptr_t)b.data_ptr() | (uintptr_t)c.data_ptr()) & 15) return {as_bf16(a), as_bf16(b), as_bf16(c)};
    auto up8 = [](int64_t x) { return (x + 7) / 8 * 8; };
    const int64_t na = a.numel(), nb = b.numel(), nc = c.numel(), ob = up8(na), oc = ob + up8(nb);
    const Tensor buf = empty({oc + up8(nc)}, at::kBFloat16, a);
    IndexInputs r{buf.narrow(0, 0, na).view(a.sizes()), buf.narrow(0, ob, nb).view(b.sizes()), buf.narrow(0, oc, nc).view(c.sizes())};
    check(dsa_round_bf16_x3(fptr(a), fptr(b), fptr(c), na, nb, nc, ptr(r.q), ptr(r.k), ptr(r.w), stream_of(a)), "dsa_round_bf16_x3");
    return r;
}

double index_scale_of(std::optional<double> s, int64_t Hi, int64_t Di) {
    return s ? *s : std::pow((double)Di, -0.5) * std::pow((double)Hi, -0.5);
}

struct Selection { Tensor idx, n, scores; };
// selection of every row; `bitmap` (may be undefined) receives the inverted selection, alone without want_list
Selection select_keys(const Tensor &qi, const Tensor &ki, const Tensor &wi, const Tensor &cu, int max_seqlen, int64_t K, double scale,
                      bool want_scores, const Tensor &bitmap, bool want_list = true) {
    TORCH_CHECK_VALUE(qi.dim() == 3 && ki.dim() == 2 && wi.dim() == 2, "indexer tensors must be q_idx (T,Hi,Di), k_idx (T,Di), w_idx (T,Hi)");
    const int64_t T = qi.size(0), Hi = qi.size(1), Di = qi.size(2);
    TORCH_CHECK_VALUE(ki.size(0) == T && ki.size(1) == Di && wi.size(0) == T && wi.size(1) == Hi, "indexer tensor shapes disagree");
    TORCH_CHECK_VALUE(K >= 1, "top_k must be >= 1");
    Selection s;
    if (want_list) {
        s.idx = empty({T, K}, at::kInt, qi);
        s.n = empty({T}, at::kInt, qi);
    }
    if (want_scores) s.scores = empty({T, K}, at::kFloat, qi);
    const size_t ws_bytes = (max_seqlen > K || want_scores) ? dsa_index_topk_workspace_bytes((int)T, max_seqlen, (int)K) : 0;
    const Tensor ws = empty_bytes(ws_bytes, qi);
    const IndexInputs in = index_inputs(qi, ki, wi);
    int32_t *idx = const_cast<int32_t *>(iptr(s.idx)), *n = const_cast<int32_t *>(iptr(s.n));
    const int N = (int)cu.numel() - 1;
    if (!want_list)
        check(dsa_index_topk_words(ptr(in.q), ptr(in.k), ptr(in.w), iptr(cu), (int)T, N, (int)Hi, (int)Di, (int)K, (float)scale, DSA_DTYPE_BF16,
                                   max_seqlen, ptr(bitmap), (size_t)bitmap.numel(), ptr(ws), ws_bytes, stream_of(qi)), "dsa_index_topk_words");
    else if (bitmap.defined())
        check(dsa_index_topk_bitmap(ptr(in.q), ptr(in.k), ptr(in.w), iptr(cu), (int)T, N, (int)Hi, (int)Di, (int)K, (float)scale, DSA_DTYPE_BF16,
                                    max_seqlen, idx, n, fptr(s.scores), ptr(bitmap), (size_t)bitmap.numel(), ptr(ws), ws_bytes, stream_of(qi)),
              "dsa_index_topk_bitmap");
    else if (want_scores)
        check(dsa_index_topk_scores(ptr(in.q), ptr(in.k), ptr(in.w), iptr(cu), (int)T, N, (int)Hi, (int)Di, (int)K, (float)scale, DSA_DTYPE_BF16,
                                    max_seqlen, idx, n, fptr(s.scores), ptr(ws), ws_bytes, stream_of(qi)), "dsa_index_topk_scores");
    else
        check(dsa_index_topk(ptr(in.q), ptr(in.k), ptr(in.w), iptr(cu), (int)T, N, (int)Hi, (int)Di, (int)K, (float)scale, DSA_DTYPE_BF16,
                             max_seqlen, idx, n, ptr(ws), ws_bytes, stream_of(qi)), "dsa_index_topk");
    return s;
}

// ---- the attention node -----------------------------------------------------------------------------------------
// bf16 inputs go to the kernels as they are.  fp32 inputs with 4*D <= 256 are carried as split-bf16 operands (x = hi + lo)
// stacked along head_dim, which keeps near-fp32 logits on the bf16 MFMA path:
//     Q' = [q_hi, q_lo, q_hi, 0]   K' = [k_hi, k_hi, k_lo, 0]   ->  Q'.K' = q.k - q_lo.k_lo
//     V' = [v_hi, v_lo, v_hi, 0]   ->  out = out'[0:D] + out'[D:2D]
//     dO' = [g_hi, g_hi, g_lo, 0]  ->  dO'.V' = g.v - g_lo.v_lo ;  dq = dq'[0:D] + dq'[2D:3D],
//                                      dk = dk'[0:D] + dk'[D:2D], dv = dv'[0:D] + dv'[2D:3D]
// Other dtypes / larger head_dim are rounded to bf16 once.
struct AttnArgs {
    int64_t max_seqlen;
    double scale;
    bool causal, want_mass, split;
    at::ScalarType dtype;
    int64_t words_k;                                     // keys per row of a selection whose bitmap is all that attention reads, else 0
};
bool carried_split(at::ScalarType dtype, int64_t D) { return dtype == at::kFloat && 4 * D <= 256; }
int rows_code(bool split, int D) { return split && D == 256 ? DSA_DTYPE_SPLIT_BF16 : DSA_DTYPE_BF16; }

void attn_forward_kernels(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &idx, const Tensor &n, const Tensor &cu, const AttnArgs &a,
                          const Tensor &ws, bool bitmap_ready, const Tensor &out, const Tensor &lse) {
    const int T = (int)q.size(0), Hq = (int)q.size(1), D = (int)q.size(2), Hkv = (int)k.size(1), N = (int)cu.numel() - 1;
    const int K = idx.defined() ? (int)idx.size(1) : 0;
    const size_t ws_bytes = ws.defined() ? (size_t)ws.numel() : 0;
    if (!idx.defined() && !a.words_k && D % 64)          // rows between the kernels' head_dims, read where they lie
        check(dsa_dense_fwd_strided(ptr(q), q.stride(0), D, ptr(k), k.stride(0), D, ptr(v), v.stride(0), D, iptr(cu), T, N, Hq, Hkv, D, (float)a.scale,
                                    DSA_DTYPE_BF16, (int)a.max_seqlen, a.causal, ptr(out), fptr(lse), stream_of(q)), "dsa_dense_fwd_strided");
    else if (a.words_k)
        check(dsa_attn_fwd_words(ptr(q), ptr(k), ptr(v), iptr(cu), T, N, Hq, Hkv, D, (int)a.words_k, (float)a.scale, rows_code(a.split, D), (int)a.max_seqlen,
                                 ptr(out), fptr(lse), ptr(ws), ws_bytes, stream_of(q)), "dsa_attn_fwd_words");
    else if (bitmap_ready)
        check(dsa_attn_fwd_saved_bitmap(ptr(q), ptr(k), ptr(v), iptr(idx), iptr(n), iptr(cu), T, N, Hq, Hkv, D, K, (float)a.scale, rows_code(a.split, D),
                                        (int)a.max_seqlen, a.causal, ptr(out), fptr(lse), ptr(ws), ws_bytes, stream_of(q)), "dsa_attn_fwd_saved_bitmap");
    else
        check(dsa_attn_fwd(ptr(q), ptr(k), ptr(v), iptr(idx), iptr(n), iptr(cu), T, N, Hq, Hkv, D, K, (float)a.scale, rows_code(a.split, D), (int)a.max_seqlen,
                           a.causal, ptr(out), fptr(lse), ptr(ws), ws_bytes, stream_of(q)), "dsa_attn_fwd");
}

Tensor attn_mass(const Tensor &q, const Tensor &k, const Tensor &lse, const Tensor &idx, const Tensor &n, const Tensor &cu, int max_seqlen,
                 double scale, const Tensor &bitmap) {
    const int T = (int)q.size(0), Hq = (int)q.size(1), D = (int)q.size(2), Hkv = (int)k.size(1), N = (int)cu.numel() - 1, K = (int)idx.size(1);
    const Tensor mass = empty({T, K}, at::kFloat, q);
    size_t ws_bytes = dsa_attn_mass_workspace_bytes(T, N, Hq, Hkv, D, K, max_seqlen);
    if (bitmap.defined()) {
        ws_bytes -= dsa_attn_fwd_workspace_bytes(T, max_seqlen, 1);          // the partial tables alone (often nothing)
        const Tensor ws = ws_bytes ? empty_bytes(ws_bytes, q) : Tensor();
        check(dsa_attn_mass_saved_bitmap(ptr(q), ptr(k), fptr(lse), iptr(idx), iptr(n), iptr(cu), T, N, Hq, Hkv, D, K, (float)scale, DSA_DTYPE_BF16,
                                         max_seqlen, fptr(mass), ptr(bitmap), (size_t)bitmap.numel(), ptr(ws), ws_bytes, stream_of(q)),
              "dsa_attn_mass_saved_bitmap");
        return mass;
    }
    const Tensor ws = empty_bytes(ws_bytes, q);
    check(dsa_attn_mass(ptr(q), ptr(k), fptr(lse), iptr(idx), iptr(n), iptr(cu), T, N, Hq, Hkv, D, K, (float)scale, DSA_DTYPE_BF16, max_seqlen,
                        fptr(mass), ptr(ws), ws_bytes, stream_of(q)), "dsa_attn_mass");
    return mass;
}

// what the forward leaves: the node's outputs and what its backward reads
struct AttnForward { Tensor qb, kb, vb, out, lse, ws, res, mass; };
AttnForward attn_forward(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu, const Tensor &idx, const Tensor &n, const Tensor &bitmap,
                         const AttnArgs &a) {
    AttnForward f;
    const int64_t T = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
    if (a.split) {
        const Tensor qc = q.contiguous(), kc = k.contiguous(), vc = v.contiguous();
        f.qb = empty({T, Hq, 4 * D}, at::kBFloat16, q);
        const Tensor kv = empty({2, T, Hkv, 4 * D}, at::kBFloat16, q);
        f.kb = kv.select(0, 0);
        f.vb = kv.select(0, 1);
        check(dsa_split_bf16_stack_qkv(fptr(qc), fptr(kc), fptr(vc), T * Hq, T * Hkv, (int)D, ptr(f.qb), ptr(f.kb), ptr(f.vb), stream_of(q)),
              "dsa_split_bf16_stack_qkv");
    } else {
        f.qb = as_bf16(q);
        f.kb = as_bf16(k);
        f.vb = as_bf16(v);
    }
    f.out = empty({T, Hq, f.qb.size(2)}, at::kBFloat16, q);
    f.lse = empty({Hq, T}, at::kFloat, q);
    // the selection bitmap - left by the top-k kernel (`bitmap`), else built by the forward - is kept for the backward
    // (with the tile crossover at 0 no kernel reads one)
    const bool tiles = a.words_k || (idx.defined() && dsa_get_tile_crossover() > 0);
    if (tiles) f.ws = bitmap.defined() ? bitmap : empty_bytes(dsa_attn_fwd_workspace_bytes((int)T, (int)a.max_seqlen, 1), q);
    attn_forward_kernels(f.qb, f.kb, f.vb, idx, n, cu, a, f.ws, tiles && bitmap.defined(), f.out, f.lse);
    if (a.split) {
        f.res = empty({T, Hq, D}, at::kFloat, q);
        check(dsa_split_bf16_combine(ptr(f.out), T * Hq, (int)D, 1, fptr(f.res), stream_of(q)), "dsa_split_bf16_combine");
    } else {
        f.res = a.dtype == at::kBFloat16 ? f.out : f.out.to(a.dtype);
    }
    // from the very operands and log-sum-exp of the forward, so that every row sums to one
    if (a.want_mass) f.mass = attn_mass(f.qb, f.kb, f.lse, idx, n, cu, (int)a.max_seqlen, a.scale, f.ws);
    return f;
}

class AttnNode : public torch::autograd::Function<AttnNode> {
public:
    static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu, const OptTensor &idx_,
                                 const OptTensor &n_, const OptTensor &bitmap_, int64_t max_seqlen, double scale, bool causal, bool want_mass,
                                 int64_t words_k) {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(q.device());
        const Tensor idx = idx_.value_or(Tensor()), n = n_.value_or(Tensor());
        const AttnArgs a{max_seqlen, scale, causal, want_mass, carried_split(q.scalar_type(), q.size(2)), q.scalar_type(), words_k};
        const AttnForward f = attn_forward(q, k, v, cu, idx, n, bitmap_.value_or(Tensor()), a);
        ctx->save_for_backward({f.qb, f.kb, f.vb, f.out, f.lse, cu, words_k ? Tensor() : idx, words_k ? Tensor() : n, f.ws});
        ctx->saved_data["m"] = max_seqlen;
        ctx->saved_data["s"] = scale;
        ctx->saved_data["c"] = causal;
        ctx->saved_data["t"] = (int64_t)a.dtype;
        ctx->saved_data["p"] = a.split;
        ctx->saved_data["w"] = words_k;
        if (!want_mass) return {f.res};
        ctx->mark_non_differentiable({f.mass});
        ctx->set_materialize_grads(false);               // (no (T,K) table of zeros as the mass's gradient)
        return {f.res, f.mass};
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        at::AutoDispatchBelowADInplaceOrView below;
        const variable_list s = ctx->get_saved_variables();
        const Tensor &q = s[0], &k = s[1], &v = s[2], &out = s[3], &lse = s[4], &cu = s[5], &idx = s[6], &n = s[7], &ws = s[8];
        const c10::OptionalDeviceGuard guard(q.device());
        const int max_seqlen = (int)ctx->saved_data["m"].toInt();
        const double scale = ctx->saved_data["s"].toDouble();
        const int causal = ctx->saved_data["c"].toBool();
        const auto dtype = (at::ScalarType)ctx->saved_data["t"].toInt();
        const bool split = ctx->saved_data["p"].toBool();
        const int words_k = (int)ctx->saved_data["w"].toInt();
        const int T = (int)q.size(0), Hq = (int)q.size(1), D = (int)q.size(2), Hkv = (int)k.size(1), N = (int)cu.numel() - 1;
        const int K = idx.defined() ? (int)idx.size(1) : 0;
        const Tensor g = grads[0].defined() ? grads[0] : at::zeros({T, Hq, split ? D / 4 : D}, out.options());
        Tensor db;
        if (split) {
            const Tensor gf = g.to(at::kFloat).contiguous();
            db = empty({T, Hq, D}, at::kBFloat16, q);
            check(dsa_split_bf16_stack(fptr(gf), (int64_t)T * Hq, D / 4, 1, ptr(db), stream_of(q)), "dsa_split_bf16_stack");
        } else {
            db = as_bf16(g);
        }
        Tensor dq = empty({T, Hq, D}, at::kBFloat16, q), dk = empty({T, Hkv, D}, at::kBFloat16, q), dv = empty({T, Hkv, D}, at::kBFloat16, q);
        if (!idx.defined() && !words_k && D % 64) {
            const size_t sc_bytes = dsa_attn_bwd_scratch_bytes(T, N, Hq, Hkv, D);
            const Tensor scratch = empty_bytes(sc_bytes, q);
            check(dsa_dense_bwd_rows(ptr(db), ptr(q), ptr(k), ptr(v), ptr(out), fptr(lse), iptr(cu), T, N, Hq, Hkv, D, (float)scale, DSA_DTYPE_BF16,
                                     max_seqlen, causal, ptr(dq), ptr(dk), ptr(dv), ptr(scratch), sc_bytes, stream_of(q)), "dsa_dense_bwd_rows");
        } else if (words_k) {
            const size_t sc_bytes = dsa_attn_bwd_scratch_bytes(T, N, Hq, Hkv, D);
            const Tensor scratch = empty_bytes(sc_bytes, q);
            check(dsa_attn_bwd_words(ptr(db), ptr(q), ptr(k), ptr(v), ptr(out), fptr(lse), iptr(cu), T, N, Hq, Hkv, D, words_k, (float)scale,
                                     rows_code(split, D), max_seqlen, ptr(dq), ptr(dk), ptr(dv), ptr(ws), (size_t)ws.numel(), ptr(scratch), sc_bytes,
                                     stream_of(q)), "dsa_attn_bwd_words");
        } else if (ws.defined() || !idx.defined()) {                               // the forward's bitmap is read where it lies
            const size_t sc_bytes = dsa_attn_bwd_scratch_bytes(T, N, Hq, Hkv, D);
            const Tensor scratch = empty_bytes(sc_bytes, q);
            check(dsa_attn_bwd_saved_bitmap(ptr(db), ptr(q), ptr(k), ptr(v), ptr(out), fptr(lse), iptr(idx), iptr(n), iptr(cu), T, N, Hq, Hkv, D, K,
                                            (float)scale, rows_code(split, D), max_seqlen, causal, ptr(dq), ptr(dk), ptr(dv), ptr(ws),
                                            ws.defined() ? (size_t)ws.numel() : 0, ptr(scratch), sc_bytes, stream_of(q)), "dsa_attn_bwd_saved_bitmap");
        } else {
            const size_t ws_bytes = dsa_attn_bwd_workspace_bytes(T, Hq, max_seqlen, 1);
            const Tensor w = empty_bytes(ws_bytes, q);
            check(dsa_attn_bwd(ptr(db), ptr(q), ptr(k), ptr(v), ptr(out), fptr(lse), iptr(idx), iptr(n), iptr(cu), T, N, Hq, Hkv, D, K, (float)scale,
                               rows_code(split, D), max_seqlen, causal, ptr(dq), ptr(dk), ptr(dv), ptr(w), ws_bytes, stream_of(q)), "dsa_attn_bwd");
        }
        if (split) {
            const Tensor oq = empty({T, Hq, D / 4}, at::kFloat, q), ok = empty({T, Hkv, D / 4}, at::kFloat, q), ov = empty({T, Hkv, D / 4}, at::kFloat, q);
            check(dsa_split_bf16_combine_qkv(ptr(dq), ptr(dk), ptr(dv), (int64_t)T * Hq, (int64_t)T * Hkv, D / 4, fptr(oq), fptr(ok), fptr(ov), stream_of(q)),
                  "dsa_split_bf16_combine_qkv");
            dq = oq; dk = ok; dv = ov;
        } else if (dtype != at::kBFloat16) {
            dq = dq.to(dtype); dk = dk.to(dtype); dv = dv.to(dtype);
        }
        return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

bool needs_grad(const Tensor &q, const Tensor &k, const Tensor &v) {
    return at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
}

struct Qkv { int64_t T, Hq, Hkv, D; };
Qkv checked_qkv(const Tensor &q, const Tensor &k, const Tensor &v) {
    TORCH_CHECK_VALUE(q.dim() == 3 && k.dim() == 3 && v.dim() == 3, "q, k, v must be (T, H, D)");
    const Qkv s{q.size(0), q.size(1), k.size(1), q.size(2)};
    TORCH_CHECK_VALUE(k.sizes() == v.sizes() && k.size(0) == s.T && k.size(2) == s.D, "q/k/v shapes disagree: ", q.sizes(), " ", k.sizes(), " ", v.sizes());
    TORCH_CHECK_VALUE(s.Hkv > 0 && s.Hq % s.Hkv == 0, "Hq=", s.Hq, " must be a multiple of Hkv=", s.Hkv);
    TORCH_CHECK_VALUE(q.scalar_type() == k.scalar_type() && q.scalar_type() == v.scalar_type(), "q, k, v must share a dtype");
    return s;
}

// a selection the caller holds: a (T, K) table of keys and (T) counts, int32, contiguous, beside the tensors it indexes
struct Picked { Tensor idx, n; };
Picked checked_selection(const OptTensor &idx, const OptTensor &n, int64_t T, const Tensor &beside) {
    TORCH_CHECK_VALUE(idx.has_value() == n.has_value(), "idx and n belong together");
    if (!idx) return {};
    TORCH_CHECK_VALUE(idx->dim() == 2 && idx->size(0) == T && idx->size(1) >= 1 && n->dim() == 1 && n->size(0) == T && idx->scalar_type() == at::kInt &&
                      n->scalar_type() == at::kInt, "a selection is idx (T,K) int32 and n (T,) int32 for T=", T, ", got ", idx->sizes(), " ",
                      idx->scalar_type(), " and ", n->sizes(), " ", n->scalar_type());
    TORCH_CHECK_VALUE(idx->device() == beside.device() && n->device() == beside.device(), "idx and n must lie on ", beside.device());
    return {idx->contiguous(), n->contiguous()};
}

variable_list attn_node(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu_, int64_t max_seqlen, const OptTensor &idx_,
                        const OptTensor &n_, double scale, bool causal, bool want_mass, const OptTensor &bitmap,
                        int64_t words_k = 0) {
    no_forward_mode({&q, &k, &v}, "attention");
    need_gpu(q); need_gpu(k); need_gpu(v); need_gpu(cu_);
    const Qkv sh = checked_qkv(q, k, v);
    TORCH_CHECK_VALUE(k.device() == q.device() && v.device() == q.device(), "q, k, v must lie on one device");
    const c10::OptionalDeviceGuard guard(q.device());
    const Tensor cu = checked_cu(cu_);
    const Picked sel = checked_selection(idx_, n_, sh.T, q);
    const OptTensor idx = sel.idx.defined() ? OptTensor(sel.idx) : std::nullopt, n = sel.n.defined() ? OptTensor(sel.n) : std::nullopt;
    TORCH_CHECK_VALUE(idx || words_k || (!want_mass && !bitmap), "the attention mass and the bitmap belong to a selection");
    TORCH_CHECK_VALUE(!bitmap || (bitmap->scalar_type() == at::kByte && bitmap->is_contiguous() && bitmap->device() == q.device()),
                      "the bitmap must be contiguous bytes on ", q.device());
    if (!needs_grad(q, k, v)) {
        at::AutoDispatchBelowADInplaceOrView below;
        const AttnArgs a{max_seqlen, scale, causal, want_mass, carried_split(q.scalar_type(), q.size(2)), q.scalar_type(), words_k};
        AttnForward f = attn_forward(q, k, v, cu, idx.value_or(Tensor()), n.value_or(Tensor()), bitmap.value_or(Tensor()), a);
        return want_mass ? variable_list{f.res, f.mass} : variable_list{f.res};
    }
    return AttnNode::apply(q, k, v, cu, idx, n, bitmap, max_seqlen, scale, causal, want_mass, words_k);
}

// q, k and v can go to the dense forward as they lie in memory: no transposing copy, no padding of the head_dim
bool readable_in_place(const Tensor &t) {
    return t.scalar_type() == at::kBFloat16 && t.stride(2) == 1 && t.size(2) % 8 == 0 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
           t.stride(0) < (1 << 24) && aligned16(t);
}
// the dense forward without a graph
Tensor dense_forward(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu, int64_t max_seqlen, double scale, bool causal) {
    const Qkv s{q.size(0), q.size(1), k.size(1), q.size(2)};
    const Tensor out = empty({s.T, s.Hq, s.D}, at::kBFloat16, q), lse = empty({s.Hq, s.T}, at::kFloat, q);
    check(dsa_dense_fwd_strided(ptr(q), q.stride(0), q.stride(1), ptr(k), k.stride(0), k.stride(1), ptr(v), v.stride(0), v.stride(1), iptr(cu), (int)s.T,
                                (int)cu.numel() - 1, (int)s.Hq, (int)s.Hkv, (int)s.D, (float)scale, DSA_DTYPE_BF16, (int)max_seqlen, causal, ptr(out),
                                fptr(lse), stream_of(q)), "dsa_dense_fwd_strided");
    return out;
}

// The same for an HF module's (1, H, T, D) tensors, (1, T, Hq, D) out: every view and check of that call in one place (a short
// generation-time batch spends 8 us on the GPU, and the views, wrappers and checks in Python took the host 15).  Nothing where
// the general path has to be taken.
std::optional<Tensor> hf_dense_forward(const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &mask, std::optional<int64_t> max_seqlen) {
    auto fits = [](const Tensor &t) {
        return t.dim() == 4 && t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.size(0) == 1 && t.stride(3) == 1 && t.size(3) % 8 == 0 &&
               t.stride(1) % 8 == 0 && t.stride(2) % 8 == 0 && t.stride(2) < (1 << 24) && aligned16(t);
    };
    if (!fits(q) || !fits(k) || !fits(v) || !mask.is_cuda() || needs_grad(q, k, v) || has_tangent(q) || has_tangent(k) || has_tangent(v) ||
        std::getenv("DSA_DEBUG_META"))
        return std::nullopt;
    const int64_t Hq = q.size(1), Hkv = k.size(1), T = q.size(2), D = q.size(3);
    if (k.sizes() != v.sizes() || k.size(2) != T || k.size(3) != D || D > 256 || !Hkv || Hq % Hkv) return std::nullopt;
    const c10::OptionalDeviceGuard guard(q.device());
    const Tensor cu = checked_cu(mask.dim() == 1 ? mask : mask.squeeze());
    const Tensor out = empty({1, T, Hq, D}, at::kBFloat16, q), lse = empty({Hq, T}, at::kFloat, q);
    check(dsa_dense_fwd_strided(ptr(q), q.stride(2), q.stride(1), ptr(k), k.stride(2), k.stride(1), ptr(v), v.stride(2), v.stride(1), iptr(cu), (int)T,
                                (int)cu.numel() - 1, (int)Hq, (int)Hkv, (int)D, (float)std::pow((double)D, -0.5), DSA_DTYPE_BF16,
                                (int)max_seqlen.value_or(T), 1, ptr(out), fptr(lse), stream_of(q)), "dsa_dense_fwd_strided");
    return out;
}

// the operator: out [, idx, n] [, mass] [, scores]
variable_list varlen_attn(const Tensor &q_, const Tensor &k_, const Tensor &v_, const Tensor &cu_, std::optional<int64_t> max_seqlen_,
                          const OptTensor &iq, const OptTensor &ik, const OptTensor &iw, std::optional<int64_t> top_k, std::optional<double> index_scale,
                          std::optional<double> softmax_scale, bool return_indices, bool causal, bool return_mass, bool return_scores) {
    no_forward_mode({&q_, &k_, &v_}, "dsa_varlen_attn");
    need_gpu(q_); need_gpu(k_); need_gpu(v_); need_gpu(cu_);
    const Qkv sh = checked_qkv(q_, k_, v_);
    const c10::OptionalDeviceGuard guard(q_.device());
    const int64_t max_seqlen = max_seqlen_.value_or(sh.T);
    const Tensor cu = checked_cu(cu_);
    const double scale = softmax_scale ? *softmax_scale : std::pow((double)sh.D, -0.5);
    const bool sparse = iq || ik || iw;
    TORCH_CHECK_VALUE(causal || !sparse, "DSA key selection is defined for causal attention only");
    int64_t d_kernel = 0;
    for (const int64_t d : {64, 96, 128, 256})           // head_dim 96 only without a key selection
        if (d >= sh.D && !(sparse && d == 96)) { d_kernel = d; break; }
    Selection sel;
    Tensor bitmap;
    int64_t words_k = 0;
    if (sparse) {
        TORCH_CHECK_VALUE(iq && ik && iw && top_k, "DSA needs indexer_q, indexer_k, indexer_w and top_k together");
        TORCH_CHECK_VALUE(iq->dim() >= 1 && iq->size(0) == sh.T, "indexer tensors must cover the same T packed tokens as q");
        need_gpu(*iq); need_gpu(*ik); need_gpu(*iw);
        at::AutoDispatchBelowADInplaceOrView below;
        // the top-k kernel leaves the inverted selection here: forward and backward read it, nothing builds it again
        if (dsa_get_tile_crossover() > 0) bitmap = empty_bytes(dsa_attn_fwd_workspace_bytes((int)sh.T, (int)max_seqlen, 1), q_);
        TORCH_CHECK_VALUE(iq->dim() == 3, "indexer tensors must be q_idx (T,Hi,Di), k_idx (T,Di), w_idx (T,Hi)");
        // ... alone, unless some row is one for the kernels that gather by the list; nothing writes a list then that the caller did not ask for
        if (bitmap.defined() &&
            !dsa_attn_batch_reads_list((int)sh.Hq, (int)sh.Hkv, (int)(carried_split(q_.scalar_type(), d_kernel) ? 4 * d_kernel : d_kernel), (int)*top_k,
                                       (int)sh.T, (int)cu.numel() - 1, (int)max_seqlen))
            words_k = *top_k;
        sel = select_keys(*iq, *ik, *iw, cu, (int)max_seqlen, *top_k, index_scale_of(index_scale, iq->size(1), iq->size(2)), return_scores, bitmap,
                          !words_k || return_indices || return_mass || return_scores);
    } else {
        TORCH_CHECK_VALUE(!return_indices && !return_scores, "return_indices / return_scores need the indexer inputs");
    }
    TORCH_CHECK_VALUE(d_kernel, "head_dim ", sh.D, " is beyond the kernels' largest (256)");
    TORCH_CHECK_VALUE(sparse || !return_mass, "return_mass needs the indexer inputs");
    Tensor q = q_, k = k_, v = v_;
    if (!sparse && !needs_grad(q, k, v) && readable_in_place(q) && readable_in_place(k) && readable_in_place(v))
        return {dense_forward(q, k, v, cu, max_seqlen, scale, causal)};
    // the tile kernels take rows of any multiple of 8 up to 128 where they lie (a selection's kernels do not)
    if (!sparse && q.scalar_type() == at::kBFloat16 && sh.D <= 128 && sh.D % 8 == 0) d_kernel = sh.D;
    if (d_kernel != sh.D) {
        // zero columns change neither q.k nor the used part of p.v
        const int64_t pad = d_kernel - sh.D;
        q = at::constant_pad_nd(q, {0, pad}); k = at::constant_pad_nd(k, {0, pad}); v = at::constant_pad_nd(v, {0, pad});
    }
    variable_list r = attn_node(q.contiguous(), k.contiguous(), v.contiguous(), cu, max_seqlen, sel.idx.defined() ? OptTensor(sel.idx) : std::nullopt,
                                sel.n.defined() ? OptTensor(sel.n) : std::nullopt, scale, causal, return_mass,
                                bitmap.defined() ? OptTensor(bitmap) : std::nullopt, words_k);
    variable_list res{d_kernel != sh.D ? r[0].narrow(-1, 0, sh.D) : r[0]};
    if (return_indices) { res.push_back(sel.idx); res.push_back(sel.n); }
    if (return_mass) res.push_back(r[1]);
    if (return_scores) res.push_back(sel.scores);
    return res;
}

// ---- the indexer's training loss ---------------------------------------------------------------------------------
struct IndexerGrads { Tensor dq, dk, dw; };
IndexerGrads indexer_bwd(const Tensor &q_idx, const Tensor &k_idx, const Tensor &w_idx, const Tensor &idx, const Tensor &n, const Tensor &dscore_,
                         const Tensor &grad, const Tensor &cu, int64_t max_seqlen, std::optional<double> index_scale) {
    const int64_t T = q_idx.size(0), Hi = q_idx.size(1), Di = q_idx.size(2), K = idx.size(1);
    const double scale = index_scale_of(index_scale, Hi, Di);
    IndexInputs in = index_inputs(q_idx, k_idx, w_idx);
    const int64_t d_kernel = Di <= 64 ? 64 : Di <= 128 ? 128 : Di;
    if (d_kernel != Di) {                                // e.g. 32-wide index heads: zero columns change no score
        in.q = at::constant_pad_nd(in.q, {0, d_kernel - Di});
        in.k = at::constant_pad_nd(in.k, {0, d_kernel - Di});
    }
    const Tensor dscore = dscore_.contiguous();
    IndexerGrads g{empty({T, Hi, d_kernel}, at::kBFloat16, in.q), empty({T, d_kernel}, at::kBFloat16, in.q),
                   empty({T, Hi}, w_idx.scalar_type() == at::kBFloat16 ? at::kBFloat16 : at::kFloat, in.q)};
    const size_t ws_bytes = dsa_indexer_bwd_workspace_bytes((int)T, (int)d_kernel, (int)max_seqlen);
    const Tensor ws = empty_bytes(ws_bytes, in.q);
    check(dsa_indexer_bwd_scaled(ptr(in.q), ptr(in.k), ptr(in.w), iptr(idx), iptr(n), fptr(dscore), fptr(grad), iptr(cu), (int)T, (int)cu.numel() - 1, (int)Hi,
                          (int)d_kernel, (int)K, (float)scale, DSA_DTYPE_BF16, (int)max_seqlen, ptr(g.dq), ptr(g.dk), ptr(g.dw),
                          g.dw.scalar_type() == at::kBFloat16 ? DSA_DTYPE_BF16 : DSA_DTYPE_FP32, ptr(ws), ws_bytes, stream_of(in.q)), "dsa_indexer_bwd_scaled");
    if (d_kernel != Di) {
        g.dq = g.dq.narrow(-1, 0, Di).contiguous();
        g.dk = g.dk.narrow(-1, 0, Di).contiguous();
    }
    return g;
}

class IndexerKLNode : public torch::autograd::Function<IndexerKLNode> {
public:
    static Tensor forward(AutogradContext *ctx, const Tensor &q_idx, const Tensor &k_idx, const Tensor &w_idx, const Tensor &mass_, const Tensor &cu,
                          const OptTensor &idx_, const OptTensor &n_, const OptTensor &sel_, int64_t max_seqlen, int64_t top_k,
                          std::optional<double> index_scale) {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(q_idx.device());
        const int64_t T = q_idx.size(0);
        TORCH_CHECK_VALUE(k_idx.size(0) == T && k_idx.size(1) == q_idx.size(2) && w_idx.size(0) == T && w_idx.size(1) == q_idx.size(1),
                          "indexer tensor shapes disagree: ", q_idx.sizes(), " ", k_idx.sizes(), " ", w_idx.sizes());
        Selection s;
        if (sel_) {
            TORCH_CHECK_VALUE(idx_ && n_, "a selection is (idx, n, scores)");
            const Picked p = checked_selection(idx_, n_, T, q_idx);
            TORCH_CHECK_VALUE(p.idx.sizes() == sel_->sizes(), "idx must have the shape of the scores: ", p.idx.sizes(), " ", sel_->sizes());
            s = {p.idx, p.n, *sel_};
        } else s = select_keys(q_idx, k_idx, w_idx, cu, (int)max_seqlen, top_k, index_scale_of(index_scale, q_idx.size(1), q_idx.size(2)), true, Tensor());
        const int64_t K = s.scores.size(1);
        TORCH_CHECK_VALUE(mass_.sizes() == s.scores.sizes() && s.scores.scalar_type() == at::kFloat && mass_.scalar_type() == at::kFloat,
                          "sel_scores and mass must be (T,K) fp32");
        TORCH_CHECK_VALUE(s.scores.device() == q_idx.device() && mass_.device() == q_idx.device(), "sel_scores and mass must lie on ", q_idx.device());
        const Tensor sc = s.scores.contiguous(), mass = mass_.contiguous();
        const Tensor loss = empty({T}, at::kFloat, q_idx), dscore = empty({T, K}, at::kFloat, q_idx);
        check(dsa_indexer_kl(fptr(sc), fptr(mass), iptr(s.n), (int)T, (int)K, 1.f / (float)std::max<int64_t>(T, 1), fptr(loss), fptr(dscore),
                             stream_of(q_idx)), "dsa_indexer_kl");
        ctx->save_for_backward({q_idx, k_idx, w_idx, s.idx, s.n, dscore, cu});
        ctx->saved_data["m"] = max_seqlen;
        if (index_scale) ctx->saved_data["s"] = *index_scale;
        return loss.mean();
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        at::AutoDispatchBelowADInplaceOrView below;
        const variable_list s = ctx->get_saved_variables();
        const c10::OptionalDeviceGuard guard(s[0].device());
        std::optional<double> scale;
        const auto it = ctx->saved_data.find("s");
        if (it != ctx->saved_data.end()) scale = it->second.toDouble();
        // the gradients are linear in dscore: the kernels multiply their sums by the incoming gradient
        const IndexerGrads g = indexer_bwd(s[0], s[1], s[2], s[3], s[4], s[5], grads[0].to(at::kFloat).contiguous(), s[6], ctx->saved_data["m"].toInt(), scale);
        return {g.dq.to(s[0].scalar_type()), g.dk.to(s[1].scalar_type()), g.dw.to(s[2].scalar_type()), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(),
                Tensor(), Tensor(), Tensor()};
    }
};

Tensor indexer_kl_loss(const Tensor &q_idx, const Tensor &k_idx, const Tensor &w_idx, const Tensor &mass, const Tensor &cu_, int64_t max_seqlen,
                       int64_t top_k, std::optional<double> index_scale, const OptTensor &idx, const OptTensor &n, const OptTensor &sel) {
    no_forward_mode({&q_idx, &k_idx, &w_idx, &mass}, "indexer_kl_loss");
    need_gpu(q_idx); need_gpu(k_idx); need_gpu(w_idx); need_gpu(mass); need_gpu(cu_);
    TORCH_CHECK_VALUE(q_idx.dim() == 3 && k_idx.dim() == 2 && w_idx.dim() == 2, "indexer tensors must be q_idx (T,Hi,Di), k_idx (T,Di), w_idx (T,Hi)");
    const c10::OptionalDeviceGuard guard(q_idx.device());
    const Tensor cu = checked_cu(cu_);
    return IndexerKLNode::apply(q_idx, k_idx, w_idx, mass, cu, idx, n, sel, max_seqlen, top_k, index_scale);
}

// ---- norm + rotation in front of the attention, gate behind it ------------------------------------------------------
void check_thd(const Tensor &x, const char *name) {
    TORCH_CHECK_VALUE(x.dim() == 3 && x.stride(2) == 1, name, " must be a (T, H, D) view with a contiguous last dimension");
    TORCH_CHECK_VALUE(x.scalar_type() == at::kBFloat16, name, " must be bf16");
}

class QkNormRopeNode : public torch::autograd::Function<QkNormRopeNode> {
public:
    static variable_list forward(AutogradContext *ctx, const Tensor &q, const Tensor &k, const Tensor &q_weight, const Tensor &k_weight, const Tensor &cos_,
                                 const Tensor &sin_, double eps, bool offset) {
        at::AutoDispatchBelowADInplaceOrView below;
        for (const Tensor *t : {&q, &k, &q_weight, &k_weight, &cos_, &sin_}) need_gpu(*t);
        TORCH_CHECK_VALUE(q.dim() == 3 && k.dim() == 3, "q, k must be (T, H, D) views");
        const c10::OptionalDeviceGuard guard(q.device());
        const int64_t T = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
        TORCH_CHECK_VALUE(k.size(0) == T && k.size(2) == D, "q/k shapes disagree: ", q.sizes(), " ", k.sizes());
        check_thd(q, "q");
        check_thd(k, "k");
        Tensor cs = cos_, sn = sin_;
        if (cs.dim() == 3 && cs.size(0) == 1) { cs = cs.select(0, 0); sn = sn.select(0, 0); }
        TORCH_CHECK_VALUE(cs.dim() == 2 && cs.sizes() == sn.sizes() && cs.size(0) == T, "cos, sin must be (T, R) or (1, T, R)");
        TORCH_CHECK_VALUE((cs.scalar_type() == at::kBFloat16 || cs.scalar_type() == at::kFloat) && sn.scalar_type() == cs.scalar_type(),
                          "cos, sin must both be bf16 or both fp32");
        const int cs_code = cs.scalar_type() == at::kBFloat16 ? DSA_DTYPE_BF16 : DSA_DTYPE_FP32, R = (int)cs.size(1);
        cs = cs.contiguous();
        sn = sn.contiguous();
        // the weights go in as the module holds them (fp32 master parameters, or bf16): no cast kernel in front of the call
        Tensor qw = q_weight.contiguous(), kw = k_weight.contiguous();
        if (qw.scalar_type() != kw.scalar_type() || (qw.scalar_type() != at::kFloat && qw.scalar_type() != at::kBFloat16)) {
            qw = qw.to(at::kFloat);
            kw = kw.to(at::kFloat);
        }
        TORCH_CHECK_VALUE(qw.numel() == D && kw.numel() == D, "norm weights must have head_dim elements");
        const int flags = (offset ? DSA_NORM_OFFSET : 0) | (qw.scalar_type() == at::kBFloat16 ? DSA_NORM_WEIGHT_BF16 : 0);
        const Tensor qo = empty({T, Hq, D}, at::kBFloat16, q), ko = empty({T, Hkv, D}, at::kBFloat16, q);
        const Tensor qr = empty({T, Hq}, at::kFloat, q), kr = empty({T, Hkv}, at::kFloat, q);
        check(dsa_qk_norm_rope_fwd(ptr(q), q.stride(0), q.stride(1), ptr(k), k.stride(0), k.stride(1), ptr(qw), ptr(kw), (float)eps, flags, ptr(cs), ptr(sn),
                                   cs_code, R, (int)T, (int)Hq, (int)Hkv, (int)D, ptr(qo), ptr(ko), fptr(qr), fptr(kr), stream_of(q)),
              "dsa_qk_norm_rope_fwd");
        ctx->save_for_backward({q, k, qw, kw, cs, sn, qr, kr});
        ctx->saved_data["f"] = (int64_t)flags;
        ctx->saved_data["q"] = (int64_t)q_weight.scalar_type();
        ctx->saved_data["k"] = (int64_t)k_weight.scalar_type();
        return {qo, ko};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        at::AutoDispatchBelowADInplaceOrView below;
        const variable_list s = ctx->get_saved_variables();
        const Tensor &q = s[0], &k = s[1], &qw = s[2], &kw = s[3], &cs = s[4], &sn = s[5], &qr = s[6], &kr = s[7];
        const c10::OptionalDeviceGuard guard(q.device());
        const int64_t T = q.size(0), Hq = q.size(1), D = q.size(2), Hkv = k.size(1);
        auto grad_of = [&](const Tensor &g, int64_t H) { return g.defined() ? as_bf16(g) : at::zeros({T, H, D}, q.options()); };
        const Tensor gq = grad_of(grads[0], Hq), gk = grad_of(grads[1], Hkv);
        const Tensor dq = empty({T, Hq, D}, at::kBFloat16, q), dk = empty({T, Hkv, D}, at::kBFloat16, q);
        const auto qt = (at::ScalarType)ctx->saved_data["q"].toInt(), kt = (at::ScalarType)ctx->saved_data["k"].toInt();
        const bool wide = qt != at::kBFloat16 || kt != at::kBFloat16;          // two bf16 gradients come from the kernel as they are
        const Tensor dqw = empty({D}, wide ? at::kFloat : at::kBFloat16, q), dkw = empty({D}, wide ? at::kFloat : at::kBFloat16, q);
        const size_t ws_bytes = dsa_qk_norm_rope_bwd_workspace_bytes((int)T, (int)D);
        const Tensor ws = empty_bytes(ws_bytes, q);
        const int cs_code = cs.scalar_type() == at::kBFloat16 ? DSA_DTYPE_BF16 : DSA_DTYPE_FP32;
        check(dsa_qk_norm_rope_bwd(ptr(gq), ptr(gk), ptr(q), q.stride(0), q.stride(1), ptr(k), k.stride(0), k.stride(1), ptr(qw), ptr(kw),
                                   (int)ctx->saved_data["f"].toInt() | (wide ? 0 : DSA_NORM_GRAD_BF16), ptr(cs), ptr(sn), cs_code, (int)cs.size(1), fptr(qr), fptr(kr), (int)T, (int)Hq,
                                   (int)Hkv, (int)D, ptr(dq), Hq * D, D, ptr(dk), Hkv * D, D, (float *)ptr(dqw), (float *)ptr(dkw), ptr(ws), ws_bytes, stream_of(q)),
              "dsa_qk_norm_rope_bwd");
        return {dq, dk, dqw.to(qt), dkw.to(kt), Tensor(), Tensor(),
                Tensor(), Tensor()};
    }
};

variable_list qk_norm_rope(const Tensor &q, const Tensor &k, const Tensor &qw, const Tensor &kw, const Tensor &cos, const Tensor &sin, double eps,
                           bool offset) {
    no_forward_mode({&q, &k, &qw, &kw, &cos, &sin}, "qk_norm_rope");
    return QkNormRopeNode::apply(q, k, qw, kw, cos, sin, eps, offset);
}

class SigmoidGateNode : public torch::autograd::Function<SigmoidGateNode> {
public:
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &gate) {
        at::AutoDispatchBelowADInplaceOrView below;
        need_gpu(x);
        need_gpu(gate);
        TORCH_CHECK_VALUE(x.dim() == 3 && x.is_contiguous() && x.scalar_type() == at::kBFloat16, "x must be a contiguous bf16 (T, H, D) tensor");
        TORCH_CHECK_VALUE(gate.sizes() == x.sizes(), "gate must have the shape of x");
        check_thd(gate, "gate");
        const c10::OptionalDeviceGuard guard(x.device());
        const Tensor y = empty(x.sizes(), at::kBFloat16, x);
        check(dsa_sigmoid_gate_fwd(ptr(x), ptr(gate), gate.stride(0), gate.stride(1), (int)x.size(0), (int)x.size(1), (int)x.size(2), ptr(y), stream_of(x)),
              "dsa_sigmoid_gate_fwd");
        ctx->save_for_backward({x, gate});
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        at::AutoDispatchBelowADInplaceOrView below;
        const variable_list s = ctx->get_saved_variables();
        const Tensor &x = s[0], &gate = s[1];
        const c10::OptionalDeviceGuard guard(x.device());
        const int64_t H = x.size(1), D = x.size(2);
        const Tensor gy = as_bf16(grads[0]), dx = empty(x.sizes(), at::kBFloat16, x), dgate = empty(x.sizes(), at::kBFloat16, x);
        check(dsa_sigmoid_gate_bwd(ptr(gy), ptr(x), ptr(gate), gate.stride(0), gate.stride(1), (int)x.size(0), (int)H, (int)D, ptr(dx), ptr(dgate), H * D, D,
                                   stream_of(x)), "dsa_sigmoid_gate_bwd");
        return {dx, dgate};
    }
};

// ---- a layer's projections of one input ---------------------------------------------------------------------------
// y_i = x W_i^T for every weight (library GEMMs, as separate linears would run them), the first one's output cut into its two
// interleaved halves per head when `gate_dim` is set.  The backward gets every gradient at once: it lays them side by side and
// runs ONE weight-gradient GEMM - the separate ones have 32 to 2048 output rows over a long contraction and leave most of the chip
// idle - and one input-gradient GEMM over the first `n_input` outputs (the others read the input detached), which also takes
// the place of the sums of their input gradients.  8192 tokens, 2048 wide, six projections: nine GEMMs and two sums 574 us ->
// two GEMMs and the copies 467 us (20 of them so that every weight's gradient owns its memory).  For as long as it runs the
// backward holds, beyond what separate linears would, the packed gradients (T x columns), the input's weights laid end to end and
// the weight gradients a second time: 102 + 17 + 26 MB there.
class ProjectionNode : public torch::autograd::Function<ProjectionNode> {
public:
    static variable_list forward(AutogradContext *ctx, const Tensor &x, at::TensorList weights, int64_t n_input, int64_t gate_dim) {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::OptionalDeviceGuard guard(x.device());
        variable_list saved{x}, outs;
        for (const Tensor &w : weights) {
            saved.push_back(w);
            const Tensor y = at::linear(x, w);
            if (gate_dim && outs.empty()) {
                const Tensor halves = y.view({y.size(0), -1, 2 * gate_dim});
                outs.push_back(halves.narrow(2, 0, gate_dim));
                outs.push_back(halves.narrow(2, gate_dim, gate_dim));
            } else {
                outs.push_back(y);
            }
        }
        ctx->save_for_backward(saved);
        ctx->saved_data["n"] = n_input;
        ctx->saved_data["g"] = gate_dim;
        ctx->set_materialize_grads(false);
        return outs;
    }
    // create_graph: the separate linears' gradients in operations that autograd follows
    static variable_list differentiable_backward(AutogradContext *ctx, const variable_list &s, const variable_list &grads, int64_t n_input, int64_t D) {
        const int64_t n_w = (int64_t)s.size() - 1, T = s[0].size(0);
        variable_list res(n_w + 3);
        for (int64_t i = 0, o = 0; i < n_w; ++i) {
            Tensor g = grads[o];
            if (D && i == 0) {
                Tensor b = grads[o + 1];
                if (g.defined() || b.defined()) {
                    if (!g.defined()) g = at::zeros_like(b);
                    if (!b.defined()) b = at::zeros_like(g);
                    g = at::cat({g, b}, 2).reshape({T, -1});
                }
                ++o;
            }
            ++o;
            if (!g.defined()) continue;
            if (ctx->needs_input_grad(1 + i)) res[1 + i] = at::mm(g.t(), i < n_input ? s[0] : s[0].detach());
            if (i < n_input && ctx->needs_input_grad(0)) {
                const Tensor dx = at::mm(g, s[1 + i]);
                res[0] = res[0].defined() ? res[0] + dx : dx;
            }
        }
        return res;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &x = s[0];
        const c10::OptionalDeviceGuard guard(x.device());
        if (at::GradMode::is_enabled()) return differentiable_backward(ctx, s, grads, ctx->saved_data["n"].toInt(), ctx->saved_data["g"].toInt());
        at::AutoDispatchBelowADInplaceOrView below;
        const int64_t n_w = (int64_t)s.size() - 1, n_input = ctx->saved_data["n"].toInt(), D = ctx->saved_data["g"].toInt(), T = x.size(0);
        variable_list res(n_w + 3);
        std::vector<Tensor> keep;
        std::vector<const void *> src;
        std::vector<int32_t> width, group, col, step;
        std::vector<int64_t> at_row(n_w, -1);
        variable_list input_weights;
        int64_t cols = 0, input_cols = 0;
        bool zero_fill = false;
        for (int64_t i = 0, o = 0; i < n_w; ++i) {
            const int halves = D && i == 0 ? 2 : 1;
            bool any = false, all = true;
            for (int p = 0; p < halves; ++p) (grads[o + p].defined() ? any : all) = grads[o + p].defined();
            if (any) {
                zero_fill |= !all;
                at_row[i] = cols;
                const int64_t w = s[1 + i].size(0);
                for (int p = 0; p < halves; ++p)
                    if (grads[o + p].defined()) {
                        const Tensor g = as_bf16(grads[o + p]);
                        keep.push_back(g);
                        src.push_back(ptr(g));
                        width.push_back((int32_t)(w / halves));
                        group.push_back((int32_t)(halves == 2 ? D : w));
                        col.push_back((int32_t)(cols + p * D));
                        step.push_back((int32_t)(halves == 2 ? 2 * D : w));
                    }
                cols += w;
                if (i < n_input) { input_cols = cols; input_weights.push_back(s[1 + i]); }
            }
            o += halves;
        }
        if (!cols) return res;
        Tensor g;
        if (src.size() == 1 && group[0] == width[0]) {
            g = keep[0].reshape({T, cols});
        } else {
            g = empty({T, cols}, at::kBFloat16, x);
            if (zero_fill) g.zero_();
            check(dsa_pack_columns((int)src.size(), src.data(), width.data(), group.data(), col.data(), step.data(), (int)T, ptr(g), cols, stream_of(x)),
                  "dsa_pack_columns");
        }
        if (ctx->needs_input_grad(0) && input_cols)
            res[0] = at::mm(g.narrow(1, 0, input_cols), input_weights.size() == 1 ? input_weights[0] : at::cat(input_weights));
        // the columns of the weights whose gradient somebody takes (all of them but for torch.autograd.grad)
        int64_t first = -1, last = -1;
        for (int64_t i = 0; i < n_w; ++i)
            if (at_row[i] >= 0 && ctx->needs_input_grad(1 + i)) {
                if (first < 0) first = at_row[i];
                last = at_row[i] + s[1 + i].size(0);
            }
        if (first < 0) return res;
        const Tensor dw = at::mm(g.narrow(1, first, last - first).t(), x);
        // Every weight gets a gradient of its own: autograd keeps what it is handed as .grad, and parts of one buffer would be
        // freed, saved and resized together.
        variable_list parts, own;
        for (int64_t i = 0; i < n_w; ++i)
            if (at_row[i] >= 0 && ctx->needs_input_grad(1 + i)) {
                parts.push_back(dw.narrow(0, at_row[i] - first, s[1 + i].size(0)));
                res[1 + i] = parts.back().numel() == dw.numel() ? dw : empty(parts.back().sizes(), at::kBFloat16, x);
                own.push_back(res[1 + i]);
            }
        if (parts.size() > 1) at::_foreach_copy_(own, parts);
        return res;
    }
};

variable_list project(const Tensor &x, const std::vector<Tensor> &weights, int64_t n_input, int64_t gate_dim) {
    no_forward_mode({&x}, "project");
    for (const Tensor &w : weights) no_forward_mode({&w}, "project");
    need_gpu(x);
    TORCH_CHECK_VALUE(x.dim() == 2 && x.scalar_type() == at::kBFloat16 && !weights.empty() && n_input >= 0 && n_input <= (int64_t)weights.size() &&
                      weights.size() + (gate_dim ? 1 : 0) <= DSA_PACK_MAX, "project: a (T, width) bf16 input and up to 8 outputs");
    for (const Tensor &w : weights)
        TORCH_CHECK_VALUE(w.dim() == 2 && w.size(1) == x.size(1) && w.size(0) % 8 == 0 && w.scalar_type() == at::kBFloat16 && w.device() == x.device(),
                          "project: weights must be (rows, ", x.size(1), ") bf16 with rows a multiple of 8");
    TORCH_CHECK_VALUE(!gate_dim || (gate_dim % 8 == 0 && weights[0].size(0) % (2 * gate_dim) == 0), "project: the first output must hold pairs of ", gate_dim);
    return ProjectionNode::apply(x, at::TensorList(weights), n_input, gate_dim);
}

Tensor sigmoid_gate(const Tensor &x, const Tensor &gate) {
    no_forward_mode({&x, &gate}, "sigmoid_gate");
    return SigmoidGateNode::apply(x, gate);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    const auto nogil = py::call_guard<py::gil_scoped_release>();
    m.def("varlen_attn", &varlen_attn, nogil);
    m.def("hf_dense_forward", &hf_dense_forward, nogil);
    m.def("attn_node", [](const Tensor &q, const Tensor &k, const Tensor &v, const Tensor &cu, int64_t max_seqlen, const OptTensor &idx, const OptTensor &n,
                          double scale, bool causal, bool want_mass, const OptTensor &bitmap) {
        return attn_node(q, k, v, cu, max_seqlen, idx, n, scale, causal, want_mass, bitmap);
    }, nogil);
    m.def("indexer_kl_loss", &indexer_kl_loss, nogil);
    m.def("qk_norm_rope", &qk_norm_rope, nogil);
    m.def("sigmoid_gate", &sigmoid_gate, nogil);
    m.def("project", &project, nogil);
}
