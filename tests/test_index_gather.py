"""The indexer backward's query side over the selected keys alone: edges of its 32-key tiles, padded heads, segments, short lists."""
import pytest
import torch

from tests.util import assert_close_bf16
from vlm_training_amd import ops

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("Hi,Di,lens,K", [
    (64, 128, (100,), 1), (64, 128, (99, 1, 160), 31), (33, 128, (130, 64), 32), (48, 64, (200, 3), 33), (64, 64, (257, 31), 64), (64, 128, (300, 290), 65),
    (32, 128, (500,), 97), (17, 64, (400, 130), 128), (1, 64, (130,), 5), (64, 128, (1025, 40), 350)])
def test_query_side_over_the_selected_keys(Hi, Di, lens, K):
    assert 2 * max(lens) >= (3 if Hi > 32 else 6) * K or lens == (500,)     # (one case on the other side of the line)
    print("index gather", Hi, Di, lens, K, flush=True)
    g = torch.Generator().manual_seed(Hi + Di + K)
    T, cu = sum(lens), [0]
    for n in lens:
        cu.append(cu[-1] + n)
    q, k, w = (torch.randn(*s, generator=g).mul_(0.5).bfloat16() for s in ((T, Hi, Di), (T, Di), (T, Hi)))
    idx = torch.full((T, K), -1, dtype=torch.int32)
    n = torch.zeros(T, dtype=torch.int32)
    want_q, want_w, scale = torch.zeros(T, Hi, Di, dtype=torch.float64), torch.zeros(T, Hi, dtype=torch.float64), Di ** -0.5
    dscore = torch.randn(T, K, generator=g)
    for s0, s1 in zip(cu, cu[1:]):
        for t in range(s0, s1):
            # any ascending list of keys up to the query, of any length
            m = min(t - s0 + 1, K if t % 3 else int(torch.randint(0, K + 1, (1,), generator=g)))
            keys = torch.randperm(t - s0 + 1, generator=g)[:m].sort().values + s0
            idx[t, :m], n[t] = keys.int(), m
            r = q[t].double() @ k[keys].double().T
            d = dscore[t, :m].double()
            want_w[t] = scale * (d * r.clamp_min(0)).sum(1)
            want_q[t] = scale * w[t].double()[:, None] * ((d * (r > 0)) @ k[keys].double())
    assert (n == 0).any() or K == 1
    ds = dscore.clone()
    ds[torch.arange(K)[None] >= n[:, None]] = float("nan")                  # (slots past n are not read)
    cu_t = torch.tensor(cu, dtype=torch.int32, device=DEV)
    dq, _, dw = ops.indexer_bwd(q.to(DEV), k.to(DEV), w.to(DEV), idx.to(DEV), n.to(DEV), ds.to(DEV), cu_t, max(lens), index_scale=scale)
    assert_close_bf16(dq, want_q.float(), "dq_idx")
    # sums of n products in fp32: n 2^-24 of their absolute sum, an element of S that rounds across zero adds less than 2^-20 of its terms
    bound = (K + 64) * 2.0 ** -24 * scale * dscore.abs().max() * (q.double().norm(dim=2) * k.double().norm(dim=1).max()) * max(K, 1) ** 0.5
    assert ((dw.double().cpu() - want_w).abs() <= bound + 1e-6).all()


@pytest.mark.gpu
@pytest.mark.parametrize("Hi,Di,K", [(64, 128, 64), (40, 64, 64), (32, 128, 32), (9, 64, 32)])
def test_a_segment_takes_its_kernel_whatever_it_is_packed_with(Hi, Di, K):
    """Selected keys alone or every tile is decided by a segment's own length (96 here): its gradients are the same to the bit in any batch
    and under any bound of the longest segment."""
    print("index gather, packed", Hi, Di, K, flush=True)
    g = torch.Generator().manual_seed(Hi + Di)
    lens = (90, 300, 95, 96, 1, 97, 33)
    T, cu = sum(lens), [0]
    for n in lens:
        cu.append(cu[-1] + n)
    q, k, w = (torch.randn(*s, generator=g).mul_(0.5).bfloat16().to(DEV) for s in ((T, Hi, Di), (T, Di), (T, Hi)))
    dscore = torch.randn(T, K, generator=g).to(DEV)

    def grads(a, b, offsets, bound):
        offs = torch.tensor(offsets, dtype=torch.int32, device=DEV)
        idx, n = ops.index_topk(q[a:b], k[a:b], w[a:b], offs, bound, K)
        dq, _, dw = ops.indexer_bwd(q[a:b], k[a:b], w[a:b], idx, n, dscore[a:b], offs, bound)
        return dq, dw

    packed, loose = grads(0, T, cu, max(lens)), grads(0, T, cu, T)
    for a, b in zip(cu, cu[1:]):
        alone = grads(a, b, [0, b - a], b - a)
        for x, y, z in zip(alone, packed, loose):
            assert torch.equal(x, y[a:b]) and torch.equal(x, z[a:b]), (a, b)
