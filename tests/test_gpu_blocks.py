"""What a workgroup does in front of and behind its tiles: finding its block among many segments, its rows of q wherever they lie, rows out."""
import math

import pytest
import torch

from tests.util import assert_close_bf16
from vlm_training_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D,Hq,Hkv,many,scale,layout", [
    (*case, layout) for case in ((64, 4, 4, True, None), (72, 6, 2, False, -0.2), (96, 3, 1, False, None), (128, 8, 2, True, None),
                                 (256, 16, 1, True, None), (256, 5, 5, False, -0.1))
    for layout in ("rows", "heads", "odd") if not (case[0] == 72 and layout == "odd")])
def test_forward_blocks(D, Hq, Hkv, many, scale, layout):
    """Segments of 0 to 90 tokens, up to 200 of them, q by tokens, by heads or (head_dims of a kernel) off 16-byte addresses;
    nothing is written past the rows that exist."""
    print("blocks", D, Hq, Hkv, many, layout, flush=True)
    g = torch.Generator().manual_seed(D + Hq)
    segs = torch.randint(0, 91, (200 if many else 7,), generator=g).tolist()
    segs[1], segs[2], T = 0, 1, sum(segs) - segs[1] - segs[2] + 1
    cu = torch.tensor([0] + segs).cumsum(0).int()
    q, k, v = (torch.randn(T, h, D, generator=g).mul_(0.5).bfloat16() for h in (Hq, Hkv, Hkv))
    lib, ms, N = _lib.load(), max(segs), len(segs)
    qd, kd, vd, cud = q.to(DEV), k.to(DEV), v.to(DEV), cu.to(DEV)
    out = torch.full(((T + 3) * Hq * D,), 7.0, dtype=torch.bfloat16, device=DEV)
    lse, s = torch.full((Hq, T), 9.0, device=DEV), torch.cuda.current_stream().cuda_stream
    sc = D ** -0.5 if scale is None else scale
    if layout == "odd":
        held = torch.empty(T * Hq * D + 8, dtype=torch.bfloat16, device=DEV)
        qd = held[3:3 + T * Hq * D].view(T, Hq, D).copy_(qd)
        rc = lib.dsa_attn_fwd(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), None, None, cud.data_ptr(), T, N, Hq, Hkv, D, 0, sc, 0, ms, 1, out.data_ptr(),
                              lse.data_ptr(), None, 0, s)
    else:
        if layout == "heads":
            qd = qd.transpose(0, 1).contiguous().transpose(0, 1)
        rc = lib.dsa_dense_fwd_strided(qd.data_ptr(), qd.stride(0), qd.stride(1), kd.data_ptr(), Hkv * D, D, vd.data_ptr(), Hkv * D, D, cud.data_ptr(), T, N,
                                       Hq, Hkv, D, sc, 0, ms, 1, out.data_ptr(), lse.data_ptr(), s)
    _lib.check(rc, "forward")
    assert bool((out[T * Hq * D:] == 7.0).all())
    got, G = out[:T * Hq * D].view(T, Hq, D).float().cpu(), Hq // Hkv
    for a, n in zip(cu.tolist(), segs):
        if n:
            x = torch.matmul(q[a:a + n].double().transpose(0, 1), k[a:a + n].double().repeat_interleave(G, 1).permute(1, 2, 0)) * sc
            x = x.masked_fill(torch.ones(n, n).triu(1).bool(), -math.inf)
            want = torch.matmul(x.softmax(-1), v[a:a + n].double().repeat_interleave(G, 1).transpose(0, 1)).transpose(0, 1)
            assert_close_bf16(got[a:a + n], want.float(), f"segment of {n}")
            torch.testing.assert_close(lse[:, a:a + n].cpu(), x.logsumexp(-1).float(), rtol=0, atol=2e-5 * math.sqrt(D))
