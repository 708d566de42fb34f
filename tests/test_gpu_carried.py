"""fp32 rows of 64 carried as bf16 rows of 256: the kernels that skip the zeros and the unread parts, against those that run all of a row."""
import pytest
import torch

from vlm_training_amd import _lib

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
