"""The host side of the operators on the device: what a call may be handed, and what it must leave alone."""
import pytest
import torch

import vlm_training_amd as M

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _randn(*shape, seed=0, grad=False):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return torch.randn(*shape, generator=g).bfloat16().to(DEV).requires_grad_(grad)


@pytest.mark.parametrize("sparse", [False, True])
def test_no_tangent_is_dropped(sparse):
    """A dual tensor that requires no gradient builds no graph; the call must refuse it all the same."""
    import torch.autograd.forward_ad as fwAD
    print("tangent", sparse, flush=True)
    T, H, D = 40, 2, 64
    cu = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    more = dict(indexer_q=_randn(T, 4, 32), indexer_k=_randn(T, 32), indexer_w=_randn(T, 4), top_k=8) if sparse else {}
    for dual in range(3):
        for no_grad in (False, True):
            with fwAD.dual_level(), torch.set_grad_enabled(not no_grad):
                qkv = [_randn(T, H, D, seed=i) for i in range(3)]
                qkv[dual] = fwAD.make_dual(qkv[dual], torch.ones_like(qkv[dual]))
                with pytest.raises(NotImplementedError):
                    M.dsa_varlen_attn(*qkv, cu, T, **more)
                if not sparse:
                    with pytest.raises(NotImplementedError):
                        M.varlen_attention_forward(*(x.transpose(0, 1).unsqueeze(0) for x in qkv), cu)
    qkv = [_randn(T, H, D, seed=i) for i in range(3)]
    with pytest.raises(RuntimeError):                     # (NotImplementedError is one)
        torch.func.jvp(lambda q: M.dsa_varlen_attn(q, *qkv[1:], cu, T, **more), (qkv[0],), (torch.ones_like(qkv[0]),))
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda q: M.dsa_varlen_attn(q, *qkv[1:], cu, T, **more))(torch.stack([qkv[0], qkv[0]]))
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda q: M.dsa_varlen_attn(q, *qkv[1:], cu, T, **more).sum())(qkv[0])
