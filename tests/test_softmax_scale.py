"""Any finite softmax_scale: zero (every selected key alike), negative (the least similar key first) and nearly zero, on every path."""
import pytest
import torch

from oracle import dsa_ref as R
from tests.util import assert_close_bf16
from vlm_training_amd import _lib, ops

DEV = "cuda"


def _reference(q, k, v, cu, scale, keep):
    """softmax(scale q k^T) v per segment in 64 bits; keep(a, b): the keys each query of segment [a, b) attends"""
    G = q.shape[1] // k.shape[1]
    out = []
    for a, b in zip(cu[:-1], cu[1:]):
        qs, ks, vs = q[a:b].transpose(0, 1), k[a:b].repeat_interleave(G, 1).transpose(0, 1), v[a:b].repeat_interleave(G, 1).transpose(0, 1)
        s = (qs @ ks.transpose(1, 2).contiguous() * scale).masked_fill(~keep(a, b), float("-inf"))
        out.append((s.softmax(-1) @ vs).transpose(0, 1))
    return torch.cat(out)


@pytest.mark.gpu
# (dq and dk, and their rounding, are proportional to the scale; the bound of assert_close_bf16 is for scales up to head_dim ** -0.5)
@pytest.mark.parametrize("scale", [0.0, -0.02, -0.0625, 1e-20, -1e-30, 1e-42])
@pytest.mark.parametrize("D,Hq,Hkv,lens,dtype", [
    (64, 4, 2, (96, 33), torch.bfloat16), (64, 12, 12, (65, 2, 160, 97) * 7, torch.bfloat16), (64, 4, 2, (64, 40), torch.float32),
    (72, 4, 4, (64, 100), torch.bfloat16), (128, 4, 2, (128, 33, 7), torch.bfloat16), (128, 16, 16, (33, 129, 160) * 6, torch.bfloat16),
    (256, 8, 2, (96, 64, 5), torch.bfloat16)])
def test_softmax_scale_of_any_sign(D, Hq, Hkv, lens, dtype, scale):
    print("scale", D, Hq, Hkv, lens, dtype, scale, flush=True)
    g = torch.Generator().manual_seed(D + Hq)
    T, cu, K = sum(lens), [0], 24
    for n in lens:
        cu.append(cu[-1] + n)
    q, k, v = (torch.randn(T, h, D, generator=g).mul_(0.5).to(dtype) for h in (Hq, Hkv, Hkv))
    do = torch.randn(T, Hq, D, generator=g).to(dtype)
    index = [torch.randn(*s, generator=g).to(torch.bfloat16).to(DEV) for s in ((T, 4, 64), (T, 64), (T, 4))]
    cu_dev = torch.tensor(cu, dtype=torch.int32, device=DEV)
    lib = _lib.load()
    for mode in ("causal", "full") if D == 72 else ("causal", "full", "selection", "gather"):
        got = [x.to(DEV).requires_grad_(True) for x in (q, k, v)]
        sel = None
        split = lib.dsa_get_tile_crossover()
        try:
            if mode == "gather":
                lib.dsa_set_tile_crossover(0)
            if mode in ("causal", "full"):
                out = ops.dsa_varlen_attn(*got, cu_dev, max(lens), softmax_scale=scale, causal=mode == "causal")
            else:
                out, idx, n, mass = ops.dsa_varlen_attn(*got, cu_dev, max(lens), indexer_q=index[0], indexer_k=index[1], indexer_w=index[2], top_k=K,
                                                        softmax_scale=scale, return_indices=True, return_mass=True)
                sel = torch.zeros(T, T + 1, dtype=torch.bool).scatter_(1, torch.where(idx < 0, T, idx).long().cpu(), True)
            out.backward(do.to(DEV))
        finally:
            lib.dsa_set_tile_crossover(split)

        def keep(a, b):
            if sel is not None:
                return sel[a:b, a:b]
            every = torch.ones(b - a, b - a, dtype=torch.bool)
            return every.tril() if mode == "causal" else every

        ref = [x.double().requires_grad_(True) for x in (q, k, v)]
        want = _reference(*ref, cu, scale, keep)
        want.backward(do.double())
        assert_close_bf16(out.detach(), want.detach().float(), f"{mode} out")
        for name, a, b in zip("qkv", got, ref):
            assert_close_bf16(a.grad, b.grad.float(), f"{mode} d{name}")
        if sel is not None:
            ref_mass = R.attention_mass(q.float(), k.float(), idx.cpu(), n.cpu(), torch.tensor(cu), scale)
            assert (mass.cpu() - ref_mass).abs().max().item() <= 2e-3, mode
        else:
            with torch.no_grad():                        # the call without a graph
                assert torch.equal(ops.dsa_varlen_attn(*got, cu_dev, max(lens), softmax_scale=scale, causal=mode == "causal"), out)
