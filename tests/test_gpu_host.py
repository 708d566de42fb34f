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


def _layer(gated, T, frozen):
    from types import SimpleNamespace
    torch.manual_seed(T)
    cfg = SimpleNamespace(hidden_size=256, num_attention_heads=4, num_key_value_heads=2, head_dim=64, rms_norm_eps=1e-6)
    m = (M.SelfAttention if gated else M.Qwen3VLTextAttention)(cfg, dsa=M.DsaConfig(index_heads=8, index_dim=64, top_k=16)).to(DEV, torch.bfloat16)
    for name, p in m.named_parameters():
        p.requires_grad_(not frozen(name))
    ang = torch.outer(torch.arange(T, device=DEV).float(), 0.1 ** torch.arange(16, device=DEV).float())
    emb = torch.cat((ang, ang), -1)
    return m, (emb.cos().bfloat16(), emb.sin().bfloat16(), torch.tensor([0, T - T // 3, T], dtype=torch.int32, device=DEV), T)


def _nodes(t):
    seen, todo = set(), [t.grad_fn]
    while todo:
        n = todo.pop()
        if n is not None and n not in seen:
            seen.add(n)
            todo += [e for e, _ in n.next_functions]
    return [n.name() for n in seen]


@pytest.mark.parametrize("gated", [False, True])
def test_frozen_projections_stay_out_of_the_graph(gated):
    print("frozen", gated, flush=True)
    T = 2048                                              # large enough for the shared node
    x = _randn(1, T, 256)
    # the indexer trained beside a frozen backbone: the layer's output has no graph, the loss reaches the indexer alone
    m, rest = _layer(gated, T, lambda n: not n.startswith("indexer."))
    y = m(x, *rest)
    assert not y.requires_grad and M.indexer_losses(m).requires_grad
    M.indexer_losses(m).backward()
    assert all((p.grad is not None) == n.startswith("indexer.") for n, p in m.named_parameters())
    # everything frozen, the input trained: no projection forms a weight gradient
    m, rest = _layer(gated, T, lambda n: True)
    xi = x.clone().requires_grad_(True)
    y = m(xi, *rest)
    assert not any("ProjectionNode" in n for n in _nodes(y))
    y.backward(torch.ones_like(y))
    assert xi.grad is not None and all(p.grad is None for p in m.parameters())
    # everything trained: the shared node is there
    m, rest = _layer(gated, T, lambda n: False)
    assert any("ProjectionNode" in n for n in _nodes(m(x, *rest)))


def test_shared_projections_form_the_gradients_that_are_taken():
    from torch.profiler import ProfilerActivity, profile
    from vlm_training_amd import _lib
    T, W = 64, 32
    x, ws = _randn(T, W, grad=True), [_randn(n, W, seed=n, grad=True) for n in (8, 16, 24)]
    gs = [_randn(T, w.shape[0], seed=7) for w in ws]
    want = torch.autograd.grad([x @ w.t() for w in ws], [x] + ws, gs)
    for take in ([0], [1], [3], [0, 2], [1, 3], [0, 1, 2, 3]):
        ys = _lib.host().project(x, ws, 3, 0)
        with profile(activities=[ProfilerActivity.CPU]) as prof:
            got = torch.autograd.grad(ys, [([x] + ws)[i] for i in take], gs)
        gemms = sum(e.count for e in prof.key_averages() if e.key == "aten::mm")
        assert gemms == (0 in take) + any(i > 0 for i in take), (take, gemms)
        for i, a in zip(take, got):
            assert a.shape == want[i].shape and (a.float() - want[i].float()).norm() <= 1e-2 * want[i].float().norm(), (take, i)


def _shifted(t):
    """The same values, contiguous, one element behind a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:].copy_(t.reshape(-1))
    return buf[1:].view(t.shape)


@pytest.mark.parametrize("D,dtype,sparse,gather", [
    (64, "bf16", True, False), (128, "bf16", True, False), (256, "bf16", True, False), (72, "bf16", False, False), (128, "bf16", False, 0),
    (256, "bf16", False, False), (64, "fp32", True, False), (128, "bf16", True, True)])
def test_views_that_start_anywhere(D, dtype, sparse, gather):
    """Contiguous views on no 16-byte boundary give the bits of aligned tensors: forward, gradients, mass, indexer's loss.
    ``gather``: with the gather kernels alone."""
    print("views", D, dtype, sparse, gather, flush=True)
    lens = (70, 33, 129)
    T, Hq, Hkv, Hi, Di, K = sum(lens), 4, 2, 8, 64, 16
    cu = torch.tensor([0, 70, 103, 232], dtype=torch.int32, device=DEV)
    dt = torch.float32 if dtype == "fp32" else torch.bfloat16
    shapes = dict(q=(T, Hq, D), k=(T, Hkv, D), v=(T, Hkv, D), dout=(T, Hq, D), iq=(T, Hi, Di), ik=(T, Di), iw=(T, Hi))
    base = {n: _randn(*s, seed=i).to(dt) for i, (n, s) in enumerate(shapes.items())}
    old = M.ops.set_tile_crossover(0) if gather else None
    try:
        res = []
        for place in (lambda t: t.clone(), _shifted):
            x = {n: place(t) for n, t in base.items()}
            assert all((t.data_ptr() & 15 == 0) == (place is not _shifted) for t in x.values())
            leaves = [x[n].requires_grad_(True) for n in ("q", "k", "v") + (("iq", "ik", "iw") if sparse else ())]
            if sparse:
                out, idx, n, mass, sel = M.dsa_varlen_attn(*leaves[:3], cu, max(lens), indexer_q=x["iq"], indexer_k=x["ik"], indexer_w=x["iw"],
                                                           top_k=K, return_indices=True, return_mass=True, return_scores=True)
                loss = M.indexer_kl_loss(*leaves[3:], mass, cu, max(lens), K, selection=(idx, n, sel))
                torch.autograd.backward((out, loss), (x["dout"], None))
                with torch.no_grad():
                    plain = M.dsa_varlen_attn(*(t.detach() for t in leaves[:3]), cu, max(lens), indexer_q=x["iq"], indexer_k=x["ik"],
                                              indexer_w=x["iw"], top_k=K)
                res.append([out, idx, n, mass, sel, loss, plain] + [t.grad for t in leaves])
            else:
                out = M.dispatch_varlen_attention(*leaves, cu, max(lens), causal=False)
                out.backward(x["dout"])
                with torch.no_grad():
                    plain = M.dispatch_varlen_attention(*(t.detach() for t in leaves), cu, max(lens))
                res.append([out, plain] + [t.grad for t in leaves])
    finally:
        if gather:
            M.ops.set_tile_crossover(old)
    for a, b in zip(*res):
        assert torch.equal(a, b)


def test_a_selection_the_caller_holds_is_checked():
    """Shapes, types and places that do not fit are refused before any launch; strided ones are copied."""
    from vlm_training_amd import _lib
    host = _lib.host()
    T, Hq, Hkv, D, Hi, Di, K = 40, 4, 2, 64, 8, 64, 16
    cu = torch.tensor([0, T], dtype=torch.int32, device=DEV)
    q, k, v = _randn(T, Hq, D), _randn(T, Hkv, D, seed=1), _randn(T, Hkv, D, seed=2)
    iq, ik, iw = _randn(T, Hi, Di, grad=True), _randn(T, Di, grad=True), _randn(T, Hi, grad=True)
    out, idx, n, mass, sel = M.dsa_varlen_attn(q, k, v, cu, T, indexer_q=iq, indexer_k=ik, indexer_w=iw, top_k=K, return_indices=True,
                                               return_mass=True, return_scores=True)

    def node(idx=idx, n=n, q=q, k=k, v=v, cu=cu, mass=False, bitmap=None):
        return host.attn_node(q, k, v, cu, T, idx, n, D ** -0.5, True, mass, bitmap)

    def loss(idx=idx, n=n, sel=sel, mass=mass, ik=ik, iw=iw):
        return M.indexer_kl_loss(iq, ik, iw, mass, cu, T, K, selection=(idx, n, sel))

    wide_idx, wide_n = torch.zeros(T, 2 * K, dtype=torch.int32, device=DEV), torch.zeros(T, 2, dtype=torch.int32, device=DEV)
    wide_idx[:, :K], wide_n[:, 1] = idx, n
    assert torch.equal(node()[0], out) and torch.equal(node(wide_idx[:, :K], wide_n[:, 1])[0], out)
    want, got = loss(), loss(wide_idx[:, :K], wide_n[:, 1])
    assert torch.equal(want, got)
    for a, b in zip(torch.autograd.grad(want, [iq, ik, iw]), torch.autograd.grad(got, [iq, ik, iw])):
        assert torch.equal(a, b)
    for bad in (dict(idx=idx[:-1]), dict(idx=idx[:, 0]), dict(idx=idx.long()), dict(n=n[:-1]), dict(n=n.long()), dict(n=n[:, None]),
                dict(idx=idx.cpu()), dict(n=n.cpu())):
        for call in (node, loss):
            with pytest.raises(ValueError):
                call(**bad)
    for bad in (dict(k=k[:-1]), dict(v=v[:, :1]), dict(q=q[..., :32]), dict(idx=None), dict(n=None), dict(idx=None, n=None, mass=True),
                dict(cu=cu[:1]), dict(q=q[:, :3]), dict(q=q.float()), dict(bitmap=torch.zeros(8, dtype=torch.int32, device=DEV))):
        with pytest.raises(ValueError):
            node(**bad)
    with pytest.raises(RuntimeError):
        node(k=k.cpu())
    for bad in (dict(sel=sel[:, :K - 1].contiguous(), mass=mass[:, :K - 1].contiguous()), dict(mass=mass[:-1]), dict(ik=ik[:-1]), dict(iw=iw[:, :4]),
                dict(ik=ik[:, :32]), dict(idx=None), dict(mass=mass.bfloat16()), dict(sel=sel.cpu())):
        with pytest.raises(ValueError):
            loss(**bad)


def test_gradients_of_shared_projections_own_their_memory():
    m, rest = _layer(True, 2048, lambda n: False)
    y = m(_randn(1, 2048, 256), *rest)
    torch.autograd.backward((y, M.indexer_losses(m)), (torch.ones_like(y), None))
    stores = [p.grad.untyped_storage() for p in m.parameters()]
    assert len({s.data_ptr() for s in stores}) == len(stores)
    assert all(s.nbytes() == p.numel() * p.element_size() for s, p in zip(stores, m.parameters()))


def _count_calls(counts, how, m):
    """Put something in front of the layer's projections that counts their calls; returns what takes it away again."""
    from torch.nn.modules import module as nnm
    lins = (m.q_proj, m.indexer.k_proj)

    def hook(mod, *args):
        if mod in lins:
            counts.append(mod)
    if how in ("register_module_forward_hook", "register_module_forward_pre_hook", "register_module_full_backward_hook",
               "register_module_full_backward_pre_hook"):
        handles = [getattr(nnm, how)(hook)]
    elif how == "forward":
        class Handle:
            def __init__(self, lin):
                self.lin, plain = lin, lin.forward
                lin.forward = lambda x: (counts.append(lin), plain(x))[1]

            def remove(self):
                del self.lin.forward
        handles = [Handle(lin) for lin in lins]
    elif how == "indexer":
        plain = m.indexer.forward
        m.indexer.forward = lambda x: (counts.append(x), counts.append(x), plain(x))[2]

        class Handle:
            def remove(self):
                del m.indexer.forward
        handles = [Handle()]
    elif how in ("class", "foreign"):
        class Other(torch.nn.Module):                     # an indexer that is none of this package's
            def __init__(self, inner):
                super().__init__()
                self.inner, self.cfg = inner, inner.cfg

            def forward(self, x):
                counts.extend((x, x))
                return self.inner(x)

        class Handle:
            def __init__(self):
                self.indexer, self.plain = m.indexer, torch.nn.Linear.forward
                if how == "foreign":
                    m.indexer = Other(m.indexer)
                else:
                    torch.nn.Linear.forward = lambda lin, x: (hook(lin), self.plain(lin, x))[1]

            def remove(self):
                m.indexer, torch.nn.Linear.forward = self.indexer, self.plain
        handles = [Handle()]
    else:
        handles = [getattr(lin, how)(hook) for lin in lins]
    return handles


@pytest.mark.parametrize("how", ["register_module_forward_hook", "register_module_forward_pre_hook", "register_module_full_backward_hook",
                                 "register_module_full_backward_pre_hook", "forward", "indexer", "class", "foreign", "register_forward_hook",
                                 "register_forward_pre_hook", "register_full_backward_hook", "register_full_backward_pre_hook"])
def test_what_stands_around_the_projections_is_run(how):
    print("around the projections", how, flush=True)
    m, rest = _layer(False, 2048, lambda n: False)
    counts = []
    handles = _count_calls(counts, how, m)
    try:
        y = m(_randn(1, 2048, 256, grad=True), *rest)
        torch.autograd.backward((y, M.indexer_losses(m)), (torch.ones_like(y), None))
    finally:
        for h in handles:
            h.remove()
    assert len(counts) == 2
    counts.clear()
    assert any("ProjectionNode" in n for n in _nodes(m(_randn(1, 2048, 256), *rest))) and not counts


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_gradients_of_the_operator_own_their_memory(dtype):
    T, Hq, Hkv, D = 40, 4, 2, 64
    q, k, v = (_randn(T, h, D, seed=i).to(dtype).requires_grad_(True) for i, h in enumerate((Hq, Hkv, Hkv)))
    M.dsa_varlen_attn(q, k, v, torch.tensor([0, T], dtype=torch.int32, device=DEV), T).sum().backward()
    stores = [t.grad.untyped_storage() for t in (q, k, v)]
    assert len({s.data_ptr() for s in stores}) == 3
    assert all(s.nbytes() == t.numel() * t.element_size() for s, t in zip(stores, (q, k, v)))


@pytest.mark.parametrize("gate", [0, 8])
def test_shared_projections_can_be_differentiated_twice(gate):
    """create_graph gives what the separate linears give, first and second gradients."""
    from vlm_training_amd import _lib
    T, W = 48, 32
    x, ws = _randn(T, W, grad=True), [_randn(n, W, seed=n, grad=True) for n in (32, 16, 24)]

    def separate(x, ws):
        ys = [h @ w.t() for h, w in zip((x, x, x.detach()), ws)]
        halves = ys[0].view(T, -1, 2 * gate).split(gate, 2) if gate else ys[:1]
        return [*halves, *ys[1:]]

    res = []
    for call in (lambda: separate(x, ws), lambda: _lib.host().project(x, ws, 2, gate)):
        for skip in (0, 1):                               # (1: without the first output or its first half)
            some = call()[skip:]
            first = torch.autograd.grad([y.float().square().sum() for y in some], [x] + ws, create_graph=True, allow_unused=True)
            second = torch.autograd.grad([g.float().square().sum() for g in first if g is not None], [x] + ws, allow_unused=True)
            res.append([*first, *second])
    for a, b in zip(res[0] + res[1], res[2] + res[3]):
        assert (a is None) == (b is None)
        if a is not None:
            # bf16 sums in another order: two roundings per product and sum, through two gradients
            assert a.shape == b.shape and (a.float() - b.float()).norm() <= 2e-2 * a.float().norm()
