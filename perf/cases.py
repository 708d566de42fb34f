"""Work that users of this package have it do, through its public entry points, for timing.

A case is a dict of plain values.  ``path`` names the call:

* ``sparse_step``     one training pass of the DSA operator: ``dsa_varlen_attn`` with indexer inputs, then ``backward``
* ``sparse_forward``  the same operator without a graph (evaluation, prefill of a packed row)
* ``indexer_step``    the operator as a DSA layer calls it while its indexer trains: selection, scores and attention mass
                      returned, ``indexer_kl_loss`` added, gradients to q, k, v and to the indexer's inputs
* ``dense_step``      dense packed attention with backward through ``dispatch_varlen_attention``: causal as the text
                      layers call it, ``causal=False`` as the vision towers do
* ``dense_forward``   ``varlen_attention_forward`` on (1, H, T, D) tensors, as the forwards installed on HF modules call it
* ``prologue_step``   the element-wise work either side of the attention: ``qk_norm_rope`` and ``sigmoid_gate`` with backward
* ``layer_step``      a whole attention layer with its own indexer (``Qwen3VLTextAttention`` / ``SelfAttention``), forward
                      and backward, every parameter gradient and the indexer's loss included

``segments`` holds the lengths of the packed segments, comma-separated; the last one may be a padding tail.  The
geometries are those of ``vlm_training_amd.workloads`` (and of the vision-tower part of ``bench.py``).
"""
import math
import random
from types import SimpleNamespace

import torch

import vlm_training_amd as V
from vlm_training_amd import workloads as W

DEV = "cuda"


def _geometry(w):
    return dict(hq=w.Hq, hkv=w.Hkv, d=w.D, hi=w.Hi, di=w.Di, top_k=w.top_k, dtype="fp32" if w.dtype == torch.float32 else "bf16",
                images=w.image_runs)


def _text(lens):
    return ",".join(str(n) for n in lens)


def _dense_geometry(w):
    return {k: v for k, v in _geometry(w).items() if k in ("hq", "hkv", "d", "dtype", "images")}


TOWER_LENS = (4096, 4096, 2304, 1024, 4096, 768)          # patches per image, as bench.py times the vision towers
HIDDEN = 2048                                             # width of the 2B models' text stack


def listed():
    c1, c2, c3, c4, c5 = W.C1, W.C2, W.C3, W.C4, W.C5
    ragged = W.random_packed_workload(c3, 16384, 11)
    return [
        # a short generation-time batch through the HF layout: two ragged segments, no gradient; launches and host work
        dict(name="dense_forward_small", path="dense_forward", segments="131,66", **_dense_geometry(c2)),
        # the fp32 toy configuration, runnable next to a CPU reference
        dict(name="sparse_step_fp32_2k", path="sparse_step", segments=_text(c1.seg_lens), **_geometry(c1)),
        # a micro-batch of a 2B text stack
        dict(name="sparse_step_8k", path="sparse_step", segments=_text(c2.seg_lens), **_geometry(c2)),
        # many short segments, head_dim 256, eight query heads per kv head
        dict(name="sparse_step_d256_16k", path="sparse_step", segments=_text(c5.seg_lens), **_geometry(c5)),
        # the headline configuration: an 8B text stack at 32 768 packed tokens
        dict(name="sparse_step_32k", path="sparse_step", segments=_text(c3.seg_lens), **_geometry(c3)),
        # one long document: scores and selection grow with the square of its length
        dict(name="sparse_step_131k", path="sparse_step", segments=_text(c4.seg_lens), **_geometry(c4)),
        # evaluation of a row packed from samples of random length (the packer's usual output: odd lengths, padding tail)
        dict(name="sparse_forward_16k", path="sparse_forward", segments=_text(ragged.seg_lens), **_geometry(c3)),
        # the indexer's training path beside the main attention at the headline configuration
        dict(name="indexer_step_32k", path="indexer_step", segments=_text(c3.seg_lens), **_geometry(c3)),
        # the operator without an indexer: what a model that does not use DSA runs in every layer
        dict(name="dense_step_32k", path="dense_step", segments=_text(c3.seg_lens), causal=True, **_dense_geometry(c3)),
        # the vision tower's call: 72-wide heads, every patch of the own image attended
        dict(name="tower_step_16k", path="dense_step", segments=_text(TOWER_LENS), causal=False, hq=16, hkv=16, d=72, dtype="bf16",
             images=False),
        # gated layers with a partial rotary width: norm + rotation in front of the attention, the gate behind it
        dict(name="prologue_step_16k", path="prologue_step", tokens=16384, hq=16, hkv=2, d=256, rotary=64),
        # a whole text layer with its indexer, projections included
        dict(name="layer_step_8k", path="layer_step", segments=_text(c2.seg_lens), hidden=HIDDEN, gated=False, rotary=128,
             **_geometry(c2)),
    ]


# ---- drawn cases -------------------------------------------------------------------------------------------------
def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _packed(rng, total, mean):
    """Log-normal sample lengths filling a row of ``total`` tokens, the rest as one padding segment."""
    lens, left = [], total
    while left > 0 and len(lens) < 200:
        n = min(int(mean * 0.67 * math.exp(rng.gauss(0.0, 0.9))) + 16, total)
        if n > left - 16:
            break
        lens.append(n)
        left -= n
    if left > 0:
        lens.append(left)
    return lens


def draw(rng: random.Random):
    path = rng.choice(("sparse_step", "sparse_step", "sparse_step", "sparse_forward", "indexer_step", "dense_step", "dense_step",
                       "dense_forward", "prologue_step", "layer_step"))
    w = rng.choice((W.C1, W.C2, W.C3, W.C5))
    if path == "prologue_step":
        hq, hkv, d, rotary = rng.choice(((16, 2, 256, 64), (16, 8, 128, 128), (32, 8, 128, 128), (8, 2, 64, 64)))
        return dict(path=path, tokens=_log_int(rng, 64, 65536), hq=hq, hkv=hkv, d=d, rotary=rotary)
    if path == "dense_forward":
        return dict(path=path, segments=_text(_packed(rng, _log_int(rng, 17, 16384), rng.choice((64, 500, 4000)))),
                    **_dense_geometry(rng.choice((W.C2, W.C3, W.C5))))
    if path == "dense_step":
        if rng.random() < 0.5:
            d, heads = rng.choice(((72, 16), (64, 16)))
            lens = _packed(rng, _log_int(rng, 256, 32768), rng.choice((700, 2500)))
            return dict(path=path, segments=_text(lens), causal=False, hq=heads, hkv=heads, d=d, dtype="bf16", images=False)
        w = rng.choice((W.C2, W.C3, W.C5))
        return dict(path=path, segments=_text(_packed(rng, _log_int(rng, 256, 65536), rng.choice((400, 1500, 6000)))), causal=True,
                    **_dense_geometry(w))
    if path == "layer_step":
        w, gated = rng.choice(((W.C2, False), (W.C5, True)))
        lens = _packed(rng, _log_int(rng, 512, 16384), rng.choice((500, 1500)))
        return dict(path=path, segments=_text(lens), hidden=HIDDEN, gated=gated, rotary=64 if gated else 128, **_geometry(w))
    if path == "sparse_step" and rng.random() < 0.25:      # one document, up to the longest
        return dict(path=path, segments=str(_log_int(rng, 8192, 131072)), **_geometry(W.C3))
    lo, hi = {W.C1: (128, 8192), W.C2: (512, 32768), W.C3: (2048, 65536), W.C5: (512, 32768)}[w]
    if path == "indexer_step":
        w = W.C2 if w is W.C1 else w
        lo, hi = 1024, 32768
    return dict(path=path, segments=_text(_packed(rng, _log_int(rng, lo, hi), rng.choice((400, 1500, 6000)))), **_geometry(w))


# ---- inputs ------------------------------------------------------------------------------------------------------
def _lens(case):
    return [int(n) for n in case["segments"].split(",")]


def _offsets(lens):
    cu = [0]
    for n in lens:
        cu.append(cu[-1] + n)
    return torch.tensor(cu, dtype=torch.int32, device=DEV)


def _dtype(case):
    return torch.float32 if case["dtype"] == "fp32" else torch.bfloat16


def _attention_inputs(case, g, sparse, leaf):
    lens = _lens(case)
    T, dt = sum(lens), _dtype(case)
    sigma = 1.0 if dt == torch.float32 else 0.5

    def normal(*shape, s=sigma):
        return torch.randn(*shape, generator=g, dtype=dt, device=DEV).mul_(s)

    t = dict(q=normal(T, case["hq"], case["d"]), k=normal(T, case["hkv"], case["d"]), v=normal(T, case["hkv"], case["d"]))
    if sparse:
        t.update(q_idx=normal(T, case["hi"], case["di"]), k_idx=normal(T, case["di"]), w_idx=normal(T, case["hi"]))
    if case.get("images"):
        # image-patch runs: rows of a run share one mean vector, so that their selections cluster
        a = 0
        for L in lens:
            for r0, r1 in ((16, 1040), (2048, 3072)):
                if L >= r1 + 1000:
                    for x in t.values():
                        x[a + r0:a + r1] += torch.randn(*x.shape[1:], generator=g, dtype=dt, device=DEV).mul_(0.5)
            a += L
    if leaf:
        t["dout"] = normal(T, case["hq"], case["d"], s=1.0)
        for name in ("q", "k", "v"):
            t[name].requires_grad_(True)
    t["cu"], t["longest"] = _offsets(lens), max(lens)
    return t


def _rope_tables(T, R, base=1e6):
    inv = 1.0 / (base ** (torch.arange(0, R, 2, dtype=torch.float32, device=DEV) / R))
    ang = torch.arange(T, dtype=torch.float32, device=DEV)[:, None] * inv[None, :]
    emb = torch.cat((ang, ang), -1)
    return emb.cos().bfloat16(), emb.sin().bfloat16()


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    path = case["path"]
    if path == "prologue_step":
        T, Hq, Hkv, D = case["tokens"], case["hq"], case["hkv"], case["d"]
        mk = lambda *s: torch.randn(*s, generator=g, dtype=torch.bfloat16, device=DEV)  # noqa: E731
        qg = mk(T, Hq, 2 * D)                             # per head [q | gate]: both halves are read in place
        s = dict(q=qg[..., :D].detach().requires_grad_(True), gate=qg[..., D:].detach().requires_grad_(True),
                 k=mk(T, Hkv, D).requires_grad_(True), x=mk(T, Hq, D).requires_grad_(True), gq=mk(T, Hq, D), gk=mk(T, Hkv, D),
                 gy=mk(T, Hq, D), qw=mk(D).mul_(0.1).requires_grad_(True), kw=mk(D).mul_(0.1).requires_grad_(True))
        s["cos"], s["sin"] = _rope_tables(T, case["rotary"])
    elif path == "layer_step":
        cfg = SimpleNamespace(hidden_size=case["hidden"], num_attention_heads=case["hq"], num_key_value_heads=case["hkv"],
                              head_dim=case["d"], rms_norm_eps=1e-6)
        dsa = V.DsaConfig(index_heads=case["hi"], index_dim=case["di"], top_k=case["top_k"])
        with torch.device(DEV):
            m = (V.SelfAttention if case["gated"] else V.Qwen3VLTextAttention)(cfg, dsa=dsa).to(torch.bfloat16)
        with torch.no_grad():
            for name, p in m.named_parameters():
                r = torch.randn(p.shape, generator=g, dtype=torch.bfloat16, device=DEV)
                p.copy_(r.mul_(0.1).add_(0.0 if case["gated"] else 1.0) if "norm" in name else r.mul_(case["hidden"] ** -0.5))
        lens = _lens(case)
        T = sum(lens)
        mk = lambda: torch.randn(1, T, case["hidden"], generator=g, dtype=torch.bfloat16, device=DEV)  # noqa: E731
        s = dict(m=m, params=list(m.parameters()), x=mk().requires_grad_(True), gy=mk(), cu=_offsets(lens), longest=max(lens))
        s["cos"], s["sin"] = _rope_tables(T, case["rotary"])
    elif path == "dense_forward":
        s = _attention_inputs(case, g, sparse=False, leaf=False)
        for name in ("q", "k", "v"):
            s[name] = s[name].transpose(0, 1).unsqueeze(0).contiguous()          # (1, H, T, D)
    else:
        s = _attention_inputs(case, g, sparse=path != "dense_step", leaf=path != "sparse_forward")
        if path == "indexer_step":
            for name in ("q_idx", "k_idx", "w_idx"):
                s[name].requires_grad_(True)
    s["path"], s["top_k"], s["causal"] = path, case.get("top_k"), case.get("causal", True)
    return s


# ---- one pass ----------------------------------------------------------------------------------------------------
def _clear(*tensors):
    for t in tensors:
        t.grad = None


def run(s):
    path = s["path"]
    if path == "sparse_step":
        q, k, v = s["q"], s["k"], s["v"]
        _clear(q, k, v)
        out = V.dsa_varlen_attn(q, k, v, s["cu"], s["longest"], indexer_q=s["q_idx"], indexer_k=s["k_idx"], indexer_w=s["w_idx"],
                                top_k=s["top_k"])
        out.backward(s["dout"])
        return [out.detach(), q.grad, k.grad, v.grad]
    if path == "sparse_forward":
        with torch.no_grad():
            return V.dsa_varlen_attn(s["q"], s["k"], s["v"], s["cu"], s["longest"], indexer_q=s["q_idx"], indexer_k=s["k_idx"],
                                     indexer_w=s["w_idx"], top_k=s["top_k"])
    if path == "indexer_step":
        q, k, v, iq, ik, iw = (s[n] for n in ("q", "k", "v", "q_idx", "k_idx", "w_idx"))
        _clear(q, k, v, iq, ik, iw)
        out, idx, n, mass, scores = V.dsa_varlen_attn(q, k, v, s["cu"], s["longest"], indexer_q=iq, indexer_k=ik, indexer_w=iw,
                                                      top_k=s["top_k"], return_indices=True, return_mass=True, return_scores=True)
        loss = V.indexer_kl_loss(iq, ik, iw, mass, s["cu"], s["longest"], s["top_k"], selection=(idx, n, scores))
        torch.autograd.backward((out, loss), (s["dout"], None))
        return [out.detach(), idx, n, mass, scores, loss.detach(), q.grad, k.grad, v.grad, iq.grad, ik.grad, iw.grad]
    if path == "dense_step":
        q, k, v = s["q"], s["k"], s["v"]
        _clear(q, k, v)
        out = V.dispatch_varlen_attention(q, k, v, s["cu"], s["longest"], causal=s["causal"])
        out.backward(s["dout"])
        return [out.detach(), q.grad, k.grad, v.grad]
    if path == "dense_forward":
        with torch.no_grad():
            return V.varlen_attention_forward(s["q"], s["k"], s["v"], s["cu"])[0]
    if path == "prologue_step":
        leaves = [s[n] for n in ("q", "k", "qw", "kw", "x", "gate")]
        _clear(*leaves)
        q, k = V.qk_norm_rope(s["q"], s["k"], s["qw"], s["kw"], s["cos"], s["sin"], offset=True)
        y = V.sigmoid_gate(s["x"], s["gate"])
        torch.autograd.backward((q, k, y), (s["gq"], s["gk"], s["gy"]))
        return [q.detach(), k.detach(), y.detach()] + [t.grad for t in leaves]
    m, x = s["m"], s["x"]
    _clear(x, *s["params"])
    y = m(x, s["cos"], s["sin"], s["cu"], s["longest"])
    loss = V.indexer_losses(m)
    torch.autograd.backward((y, loss), (s["gy"], None))
    return [y.detach(), loss.detach(), x.grad] + [p.grad for p in s["params"]]


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _pairs(case):
    """(pairs the attention has to form, pairs the indexer has to score)."""
    lens, K = _lens(case), case.get("top_k")
    if not case.get("causal", True):
        return sum(n * n for n in lens), 0
    tri = lambda n: n * (n + 1) // 2  # noqa: E731
    every = sum(tri(n) for n in lens)
    if K is None:
        return every, 0
    selected = sum(tri(min(n, K)) + max(0, n - K) * K for n in lens)
    # a row whose window holds at most K keys needs no scores - unless the indexer trains on them
    scored = every if case["path"] in ("indexer_step", "layer_step") else every - sum(tri(min(n, K)) for n in lens)
    return selected, scored


def work(case):
    path, e = case["path"], 2
    if path == "prologue_step":
        T, Hq, Hkv, D = case["tokens"], case["hq"], case["hkv"], case["d"]
        rows, gate = (Hq + Hkv) * D * e, Hq * D * e
        return {"bytes": T * (4 * rows + 6 * gate + 2 * case["rotary"] * e), "flops": 60.0 * T * (2 * Hq + Hkv) * D}
    T = sum(_lens(case))
    e = 4 if case["dtype"] == "fp32" else 2
    Hq, Hkv, D = case["hq"], case["hkv"], case["d"]
    S, P = _pairs(case)
    if path == "dense_forward":
        return {"bytes": T * 2 * (Hq + Hkv) * D * e, "flops": 4.0 * Hq * D * S}
    if path == "sparse_forward":
        Hi, Di = case["hi"], case["di"]
        return {"bytes": T * (2 * (Hq + Hkv) * D + Hi * Di + Di + Hi) * e, "flops": 4.0 * Hq * D * S + (2.0 * Hi * Di + 2 * Hi) * P}
    # forward 4, backward 10 flop per pair, head and element; q k v dO in, out and three gradients out
    nbytes, flops = T * 4 * (Hq + Hkv) * D * e, 14.0 * Hq * D * S
    if "hi" in case:
        Hi, Di, K = case["hi"], case["di"], case["top_k"]
        nbytes += T * (Hi * Di + Di + Hi) * e
        flops += (2.0 * Hi * Di + 2 * Hi) * P
        if path in ("indexer_step", "layer_step"):
            # gradients of the scores w.r.t. the indexer's inputs: 4 flop per selected pair, head and element (the scores
            # themselves are there); the mass is formed from the forward's probabilities
            flops += 4.0 * Hi * Di * S
            nbytes += T * (Hi * Di + Di + Hi) * e
        if path == "indexer_step":
            nbytes += T * K * 12
    if path == "layer_step":
        cols = (2 if case["gated"] else 1) * Hq * D + 2 * Hkv * D + Hq * D
        h = case["hidden"]
        idx_cols = case["hi"] * case["di"] + case["di"] + case["hi"]
        flops += 6.0 * T * h * cols + 4.0 * T * h * idx_cols          # the indexer's input takes no gradient
        nbytes = 4 * T * h * e + 2 * (cols + idx_cols) * h * e
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # operands, probabilities and results are bf16 (8 bits) with fp32 sums; an fp32 caller's operands are carried as two
    # bf16 parts, but the probabilities and the two parts of each result still round to bf16
    if case["path"] == "indexer_step":
        # two scores that differ in the last fp32 bit may change places at the edge of a selection
        return {"rel": 1e-2, "differ": 5e-3}
    return {"rel": 1e-2}
