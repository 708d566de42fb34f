"""Selection from rows longer than the kernel holds whole: one sweep with a sampled threshold, and the radix select where that does not
serve.  The order is total (score descending, column ascending), so that every selection is exact."""
import pytest
import torch

from vlm_training_amd import _lib

DEV = "cuda"


def _scores(kind, rows, T, ld, seed):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(rows, ld, generator=g)
    if kind == "ties":
        x = (x * 2).round() / 2
    elif kind == "equal":
        x.fill_(0.25)
    elif kind == "relu":
        x.clamp_(min=0.0).mul_((torch.rand(rows, ld, generator=g) < 0.2).float()).mul_(-1.0)      # (mostly zeros of both signs)
    elif kind == "sink":
        x[:, 0], x[:, 77] = 3e38, -3e37
    elif kind == "inf":
        x[:, 5], x[:, 9] = float("inf"), float("-inf")
    elif kind == "ramp":
        x = torch.arange(ld, dtype=torch.float32).expand(rows, ld) * 1e-3
    elif kind == "hidden":                              # the sampled runs hold none of the largest scores
        for run in range(256):
            a = run * (T - rows - 15) // 255
            x[:, max(a - rows, 0):a + 16 + rows] = -5.0
    elif kind == "late":
        x += torch.linspace(-4.0, 4.0, ld)
    return x.contiguous()


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,kind,pad", [
    (8193, 2048, "normal", 3), (8196, 1, "normal", 0), (8230, 4096, "normal", 2), (8230, 4097, "normal", 2), (9000, 2048, "ties", 0),
    (12289, 64, "sink", 3), (16390, 2048, "hidden", 2), (16384, 300, "inf", 0), (20481, 2048, "late", 7), (20000, 512, "equal", 0),
    (30003, 1000, "relu", 1), (30003, 4096, "ramp", 1), (40000, 2048, "normal", 1), (131072, 1000, "normal", 0), (131073, 100, "normal", 3),
    (131071, 777, "sink", 1)])
def test_long_rows_select_exactly(T, K, kind, pad):
    rows, ld = 24, T + pad
    print("top-k", T, K, kind, ld, flush=True)
    x = _scores(kind, rows, T, ld, T + K)
    xd, cu = x.to(DEV), torch.tensor([0, T], dtype=torch.int32, device=DEV)
    idx = torch.full((T, K), -9, dtype=torch.int32, device=DEV)
    n = torch.zeros(T, dtype=torch.int32, device=DEV)
    lib = _lib.load()
    rc = lib.dsa_topk_from_scores(xd.data_ptr(), ld, T - rows, T, cu.data_ptr(), T, 1, K, idx.data_ptr(), n.data_ptr(),
                                  torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "dsa_topk_from_scores")
    got, n = idx[T - rows:].cpu(), n[T - rows:].cpu()
    for i in range(rows):
        width = T - rows + i + 1
        want = torch.sort(x[i, :width], descending=True, stable=True).indices[:K].sort().values
        assert int(n[i]) == min(width, K) and torch.equal(got[i, :len(want)].long(), want), (i, width)
