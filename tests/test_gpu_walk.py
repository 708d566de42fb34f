"""The compacted walks (thin selections): the lines to the tile and gather kernels, the ends of blocks, lists and segments."""
import math

import pytest
import torch

from tests.util import assert_close_bf16
from vlm_training_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV, D = "cuda", 128


def _reference(q, k, v, dout, sel, scale):
    """Out, log-sum-exp and gradients in 64 bits; ``sel`` (T,T): which keys a query attends.  Rows without a key: zero, -inf."""
    q, k, v = (x.double().requires_grad_(True) for x in (q, k, v))
    G = q.shape[1] // k.shape[1]
    s = torch.einsum("thd,shd->hts", q, k.repeat_interleave(G, 1)) * scale
    s = s.masked_fill(~sel, -math.inf)
    top = s.detach().amax(-1, keepdim=True).clamp(min=-1e300)
    e = (s - top).exp()
    z = e.sum(-1, keepdim=True)
    out = torch.einsum("hts,shd->thd", e / z.clamp(min=1e-300), v.repeat_interleave(G, 1))
    out.backward(dout.double())
    return out.detach(), (top + z.log()).squeeze(-1).detach(), q.grad, k.grad, v.grad


@pytest.mark.parametrize("Hq,Hkv,lens,K,kind,scale", [
    # (heads enough for the walk to take segments from 290 tokens on, or from 150 where the segments of a batch are as long on average)
    (288, 72, (641, 256, 257, 97), 8, "random", None),   # tiles to 256, walk to 768: rows on either side of a block of 96 queries
    (296, 74, (1000, 290, 289) + (21,) * 20, 8, "random", None),      # and the gather beyond 768; segments on either side of the walk's line
    (440, 220, (1400, 300), 8, "random", None),          # two heads per kv head: the gather from 1280 on
    (80, 40, (900, 770, 768), 8, "random", None),        # fewer of them: segments longer than the tiles reach
    (288, 96, (700,), 16, "random", -0.1),               # a group of three, a negative scale
    (296, 74, (1025, 705), 40, "runs", None),             # every key of a block wanted by some query: four steps
    (288, 72, (769,), 8, "classes", None),               # keys 16 apart: one class of the block's rows
    (288, 96, (640,), 12, "empty", None)])               # queries that select nothing
def test_rows_of_the_compacted_walk(Hq, Hkv, lens, K, kind, scale):
    print("compacted walk", Hq, Hkv, lens, K, kind, flush=True)
    lib, G = _lib.load(), Hq // Hkv
    past_tiles = (75 * K + 255) // 256 * 256 + 1
    first = min(16 * K + 100000 // Hq, max(past_tiles, 16 * K + 40000 // Hq)) if G == 2 else 16 * K + 12000 // Hkv      # the shortest segment that walks
    assert lib.dsa_get_tile_crossover() == 24 and max(lens) >= max(first, (26 if G == 2 else 18) * K)
    g = torch.Generator().manual_seed(Hq * K + len(lens))
    T, cu = sum(lens), [0]
    for n in lens:
        cu.append(cu[-1] + n)
    gd = torch.Generator(device=DEV).manual_seed(Hq * K + len(lens))
    q, k, v, dout = (torch.randn(T, h, D, generator=gd, device=DEV).mul_(0.5).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    idx, n = torch.full((T, K), -1, dtype=torch.int32), torch.zeros(T, dtype=torch.int32)
    sel = torch.zeros(T, T, dtype=torch.bool)
    for a, b in zip(cu[:-1], cu[1:]):
        for t in range(a, b):
            pos = t - a
            if kind == "random" or pos < K:
                keys = torch.randperm(pos + 1, generator=g)[:K]
            elif kind == "runs":
                keys = torch.arange(K) + int(torch.randint(0, pos + 2 - K, (1,), generator=g))
            elif kind == "classes":
                keys = (torch.arange(K) * 16 + pos % 16).clamp(max=pos).unique()
            else:
                keys = torch.randperm(pos + 1, generator=g)[:K if pos % 3 else 0]
            keys = keys.sort().values + a
            n[t] = len(keys)
            idx[t, :len(keys)] = keys.int()
            sel[t, keys] = True
    scale = D ** -0.5 if scale is None else scale
    sel = sel.to(DEV)
    d = [q, k, v] + [x.to(DEV) for x in (idx, n, torch.tensor(cu, dtype=torch.int32))] + [dout]
    out, lse = ops.attn_fwd(*d[:6], max(lens), scale, True)[:2]
    # the backward takes log-sum-exps that are finite, as those of rows with a key are
    dq, dk, dv = ops.attn_bwd(d[6], *d[:3], out, lse.clamp(min=-1e30), *d[3:6], max(lens), scale, causal=True)
    torch.cuda.synchronize()
    some = (n > 0).to(DEV)
    late = torch.cat([torch.arange(m) >= 16 * K + 255 for m in lens]).to(DEV)      # (the tile kernels have no result for a row without a key)
    if kind == "empty":
        assert bool((out[late & ~some] == 0).all()) and bool((dq[late & ~some] == 0).all())
    rows = some | late
    for h in range(0, Hkv, 23):
        hs = slice(h * G, (h + 1) * G)
        want = _reference(q[:, hs], k[:, h:h + 1], v[:, h:h + 1], dout[:, hs], sel, scale)
        for name, got, ref in (("out", out[:, hs], want[0]), ("dq", dq[:, hs], want[2])):
            assert_close_bf16(got[rows], ref[rows], f"{name} of kv head {h}")
        got, ref = lse[hs].T[rows], want[1].T[rows].float()
        assert torch.equal(got.isinf(), ref.isinf()) and float((got - ref)[~ref.isinf()].abs().max()) < 2e-3   # (bf16 products are exact in fp32)
        if bool(some.all()):
            assert_close_bf16(dk[:, h:h + 1], want[3], f"dk of kv head {h}")
            assert_close_bf16(dv[:, h:h + 1], want[4], f"dv of kv head {h}")


@pytest.mark.parametrize("G,lens,kind", [
    (4, (1700, 900, 500), "random"),     # 40 K = 1600: the walk takes the first segment, the tile kernel the others
    (3, (1614, 1599), "random"),         # a group of three; 1614 keys: the last workgroup's 78, the last wave's 14
    (4, (1600, 1599), "runs"),           # every query of a block wants a key of the tile, or none does
    (8, (1921, 1200), "same"),           # sixteen keys that all queries want: large probabilities, lists that are full
    (16, (2000, 1100), "classes")])      # queries of one residue: one class of the block's rows
def test_keys_of_the_compacted_walk(G, lens, kind):
    print("compacted walk, key side", G, lens, kind, flush=True)
    Hkv, K, T, scale = 64, 40, sum(lens), D ** -0.5
    assert _lib.load().dsa_get_tile_crossover() == 24 and (T // 128 + len(lens)) * Hkv > 1536
    g = torch.Generator(device=DEV).manual_seed(G)
    q, k, v, dout = (torch.randn(T, h, D, generator=g, device=DEV).mul_(0.5).bfloat16() for h in (G * Hkv, Hkv, Hkv, G * Hkv))
    idx, n = torch.full((T, K), -1, dtype=torch.int32, device=DEV), torch.zeros(T, dtype=torch.int32, device=DEV)
    sel, a, cu = torch.zeros(T, T, dtype=torch.bool, device=DEV), 0, [0]
    for m in lens:
        r = torch.rand(m, m, generator=g, device=DEV)                  # the K largest of a row are its keys
        pos = torch.arange(m, device=DEV)
        if kind == "runs":
            r += (pos[None, :] // K == (pos[:, None] * 7 // 320) % 30).float()
        elif kind == "same":
            r += (pos[None, :] % 97 < 1).float()
        elif kind == "classes":
            r += (pos[None, :] % 16 == pos[:, None] % 4).float()
        r.masked_fill_(pos[None, :] > pos[:, None], -1.0)
        top = r.topk(min(K, m)).indices
        s = torch.zeros(m, m, dtype=torch.bool, device=DEV).scatter_(1, top, True) & (pos[None, :] <= pos[:, None])
        sel[a:a + m, a:a + m] = s
        n[a:a + m] = s.sum(1).int()
        order = torch.where(s, pos[None, :], m).sort(1).values[:, :K]
        idx[a:a + m, :order.shape[1]] = torch.where(order < m, order + a, -1).int()
        a += m
        cu.append(a)
    cu = torch.tensor(cu, dtype=torch.int32, device=DEV)
    out, lse = ops.attn_fwd(q, k, v, idx, n, cu, max(lens), scale, True)[:2]
    dq, dk, dv = ops.attn_bwd(dout, q, k, v, out, lse, idx, n, cu, max(lens), scale, causal=True)
    again = ops.attn_bwd(dout, q, k, v, out, lse, idx, n, cu, max(lens), scale, causal=True)
    torch.cuda.synchronize()
    assert all(torch.equal(x, y) for x, y in zip((dq, dk, dv), again))
    for h in range(0, Hkv, 9):
        rows = slice(h * G, (h + 1) * G)
        want = _reference(q[:, rows], k[:, h:h + 1], v[:, h:h + 1], dout[:, rows], sel, scale)
        for name, got, ref in (("out", out[:, rows], want[0]), ("dq", dq[:, rows], want[2]), ("dk", dk[:, h:h + 1], want[3]), ("dv", dv[:, h:h + 1], want[4])):
            assert_close_bf16(got, ref, f"{name} of kv head {h}")


@pytest.mark.parametrize("Hq,Hkv,lens,K,empty", [(288, 72, (1200, 60, 700), 16, False), (440, 220, (1500,), 16, True), (288, 96, (900,), 12, True)])
def test_what_a_key_holds_reaches_the_rows_that_selected_it(Hq, Hkv, lens, K, empty):
    """Inf and NaN in keys, queries and gradients: rows of the walk hold what the gather kernels give, which read a row's own keys alone."""
    print("walk, not finite", Hq, Hkv, lens, K, flush=True)
    T, cu, g = sum(lens), torch.tensor([0, *lens]).cumsum(0).int(), torch.Generator(device=DEV).manual_seed(Hkv)
    q, k, v, dout = (torch.randn(T, h, D, generator=g, device=DEV).mul_(0.5).bfloat16() for h in (Hq, Hkv, Hkv, Hq))
    idx, n, pos = torch.full((T, K), -1, dtype=torch.int32), torch.zeros(T, dtype=torch.int32), torch.cat([torch.arange(m) for m in lens])
    cg = torch.Generator().manual_seed(Hkv)
    for a, m in zip(cu.tolist(), lens):
        for p in range(m):
            keys = torch.randperm(p + 1, generator=cg)[:0 if empty and p > K and p % 5 == 0 else K].sort().values + a
            n[a + p], idx[a + p, :len(keys)] = len(keys), keys.int()
    v[100, :, 5], v[333, :, :], k[210, :, 9] = math.inf, math.nan, math.nan
    k[417, ::2, 3], v[520, 1::2, 77] = -math.inf, -math.inf
    q[600, ::3, 0], dout[640, ::5, 11] = math.inf, math.nan
    d = [x.to(DEV) for x in (idx, n, cu)]
    scale, res, old = D ** -0.5, [], _lib.load().dsa_get_tile_crossover()
    assert old == 24
    try:
        for crossover in (old, 0):
            ops.set_tile_crossover(crossover)
            out, lse = ops.attn_fwd(q, k, v, *d, max(lens), scale, True)[:2]
            if crossover:
                first = (out, lse)
            dq = ops.attn_bwd(dout, q, k, v, first[0], first[1].clamp(min=-1e30), *d, max(lens), scale, causal=True)[0]
            res.append((out, lse.T, dq))
    finally:
        ops.set_tile_crossover(old)
    late = (pos >= (16 * K + 255) // 256 * 256).to(DEV) & torch.cat([torch.full((m,), m >= 600) for m in lens]).to(DEV)
    touched = torch.isin(idx, torch.tensor([100, 333, 210, 417, 520])).any(1).to(DEV)
    touched[600] = touched[640] = True
    assert int((late & ~touched).sum()) > 100 and int((late & touched).sum()) > 20
    for name, a, b in zip(("out", "lse", "dq"), *res):
        a, b = a[late].float(), b[late].float()
        assert bool((a.isfinite() == b.isfinite()).all()), name             # (a gathered row's last key also stands behind its end, with 0: Inf turns to NaN)
        assert bool(a[~touched[late]].isfinite().all()) or name == "lse" and empty
        there = b.isfinite()
        assert_close_bf16(a[there], b[there], name)
