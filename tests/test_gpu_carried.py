"""fp32 rows of 64 carried as bf16 rows of 256: the kernels that skip the zeros and the unread parts, against those that run all of a row."""
import pytest
import torch

from vlm_training_amd import _lib, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("Hq,Hkv,segs,K,causal,scale", [
    (8, 2, (300, 65, 1, 214), 48, 1, 0.125), (4, 4, (129, 31), 200, 1, -0.3), (16, 1, (200,), 8, 1, 0.2),    # tiles, whole windows, gathered rows
    (6, 2, (1900, 97), 256, 1, 0.125),                   # walks in pieces, three heads of a group of four
    (4, 2, (500, 33), 0, 1, 0.125), (2, 1, (160, 32), 0, 0, -0.1), (8, 1, (64,), 0, 0, 0.3)])                # without a selection
def test_carried_rows_give_the_bits_of_whole_rows(Hq, Hkv, segs, K, causal, scale):
    """Skipped k-steps add zeros and skipped d-tiles are never read, so every part that is read is the same bit for bit."""
    print("carried", Hq, Hkv, segs, K, causal, flush=True)
    lib, p = _lib.load(), lambda x: None if x is None else x.data_ptr()
    g = torch.Generator().manual_seed(Hq + sum(segs) + K)
    T, N, D, ms = sum(segs), len(segs), 64, max(segs)
    cu = torch.tensor([0] + list(segs)).cumsum(0).int().to(DEV)
    stream = torch.cuda.current_stream().cuda_stream

    def carried(H, order):
        x, y = torch.randn(T, H, D, generator=g).to(DEV), torch.empty(T, H, 4 * D, dtype=torch.bfloat16, device=DEV)
        _lib.check(lib.dsa_split_bf16_stack(p(x), T * H, D, order, p(y), stream), "dsa_split_bf16_stack")
        return y
    q, k, v, do = carried(Hq, 0), carried(Hkv, 1), carried(Hkv, 0), carried(Hq, 1)
    idx = n = None
    if K:
        rows = [(a, t) for a, L in zip(cu.tolist(), segs) for t in range(L)]
        pick = [(torch.randperm(t + 1, generator=g)[:K].sort().values + a) for a, t in rows]
        n = torch.tensor([len(x) for x in pick], dtype=torch.int32, device=DEV)
        idx = torch.stack([torch.nn.functional.pad(x, (0, K - len(x)), value=-1) for x in pick]).int().to(DEV)
    got = []
    for code in (_lib.DSA_DTYPE_BF16, _lib.DSA_DTYPE_SPLIT_BF16):
        out, lse = torch.full_like(q, float("nan")), torch.empty(Hq, T, device=DEV)
        ws = torch.empty(max(lib.dsa_attn_fwd_workspace_bytes(T, ms, K > 0), 1), dtype=torch.uint8, device=DEV)
        _lib.check(lib.dsa_attn_fwd(p(q), p(k), p(v), p(idx), p(n), p(cu), T, N, Hq, Hkv, 4 * D, K, scale, code, ms, causal, p(out), p(lse), p(ws),
                                    ws.numel(), stream), "dsa_attn_fwd")
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
        ws = torch.empty(lib.dsa_attn_bwd_workspace_bytes(T, Hq, ms, K > 0), dtype=torch.uint8, device=DEV)
        _lib.check(lib.dsa_attn_bwd(p(do), p(q), p(k), p(v), p(out), p(lse), p(idx), p(n), p(cu), T, N, Hq, Hkv, 4 * D, K, scale, code, ms, causal,
                                    p(dq), p(dk), p(dv), p(ws), ws.numel(), stream), "dsa_attn_bwd")
        parts = [x.view(T, -1, 4, D) for x in (dq, dk, dv)]
        got.append((out, lse, parts[0][:, :, 0::2][:, :, :2], parts[1][:, :, :2], parts[2][:, :, 0::2][:, :, :2]))
    for whole, part in zip(*got):
        assert torch.equal(whole, part)
    assert lib.dsa_attn_fwd(p(q), p(k), p(v), p(idx), p(n), p(cu), T, N, Hq, Hkv, 128, K, scale, _lib.DSA_DTYPE_SPLIT_BF16, ms, causal, p(out), p(lse),
                            p(ws), ws.numel(), stream) == -2


@pytest.mark.parametrize("Hq,Hkv,segs,K,causal,dtype", [
    (16, 2, (700, 65, 129), 100, True, torch.bfloat16),  # a selection with whole windows; gathered rows (past 24 K) in none
    (4, 4, (1, 500), 64, True, torch.bfloat16), (6, 2, (257,), 300, True, torch.bfloat16), (16, 1, (1500, 40), 64, True, torch.bfloat16),
    (8, 4, (400, 31), None, True, torch.bfloat16), (2, 1, (128, 333), None, False, torch.bfloat16),
    (4, 1, (300, 64), 50, True, torch.float32), (2, 2, (350,), None, True, torch.float32),
    # by default one launch up to 300 000 rows, or of short segments; past that one pass after the other
    (100, 25, (1700, 1300), None, True, torch.bfloat16), (100, 25, (1701, 1300), 900, True, torch.bfloat16), (120, 30, (256,) * 10, None, True, torch.bfloat16),
    (304, 76, (1000,), None, False, torch.float32)])
def test_both_passes_in_one_launch_give_the_bits_of_two(Hq, Hkv, segs, K, causal, dtype):
    print("one launch", Hq, Hkv, segs, K, causal, dtype, flush=True)
    lib, D = _lib.load(), 256 if dtype == torch.bfloat16 else 64
    g = torch.Generator().manual_seed(Hq + sum(segs))
    T, cu = sum(segs), torch.tensor([0] + list(segs)).cumsum(0).int().to(DEV)
    mk = lambda *s: torch.randn(*s, generator=g).mul_(0.5).to(dtype).to(DEV)
    q, k, v, do = mk(T, Hq, D), mk(T, Hkv, D), mk(T, Hkv, D), mk(T, Hq, D)
    sel = dict(indexer_q=mk(T, 4, 64), indexer_k=mk(T, 64), indexer_w=mk(T, 4), top_k=K) if K else dict(causal=causal)
    res, old = [], lib.dsa_get_bwd_overlap()
    try:
        for mode in (0, 1, 2):
            _lib.check(lib.dsa_set_bwd_overlap(mode), "dsa_set_bwd_overlap")
            a, b, c = (x.clone().requires_grad_(True) for x in (q, k, v))
            ops.dsa_varlen_attn(a, b, c, cu, max(segs), **sel).backward(do)
            res.append((a.grad, b.grad, c.grad))
    finally:
        lib.dsa_set_bwd_overlap(old)
    for apart, default, one in zip(*res):
        assert torch.equal(apart, default) and torch.equal(apart, one)
