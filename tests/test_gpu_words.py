"""Selections that are there as their bitmap alone: the words, and attention read from them, are those of the path with a list."""
import pytest
import torch

from vlm_training_amd import _lib, ops, workloads as W

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("segs,K,ties", [
    ((700, 333, 40, 0, 515, 204), 256, False),           # rows inside and past top_k, an empty segment
    ((1101, 65), 64, True),                              # keys of seven kinds: the last taken score is shared by many
    ((64, 1), 1, False), ((63,), 200, False),
    ((8192, 8257), 512, False),                          # both sides of the rows that are held in LDS, swept once past them
    ((9001, 300), 512, True),                            # and handed on: more of one score than the held list takes
    ((8500,), 4100, False)])                             # past the selections of the single sweep
def test_words_alone_are_those_beside_the_list(segs, K, ties):
    print("words alone", segs, K, ties, flush=True)
    w = W.scaled(W.C2, segs, top_k=K, name="words")
    t = W.make_inputs(w, device=DEV)
    qi, ki, wi, cu, lib = t["q_idx"], t["k_idx"], t["w_idx"], t["cu_seqlens"], _lib.load()
    if ties:
        ki = ki[torch.randint(0, 7, (w.T,), generator=torch.Generator().manual_seed(K)).to(DEV)].contiguous()
    T, Hi, Di = qi.shape
    p = lambda x: x.data_ptr()
    for ms in (w.max_seqlen, w.T):
        ldw = (ms + 31) // 32
        want = torch.empty(lib.dsa_attn_fwd_workspace_bytes(T, ms, 1), dtype=torch.uint8, device=DEV)
        ops.index_topk(qi, ki, wi, cu, ms, K, bitmap=want)
        want = want[:T * ldw * 4].view(torch.int32)
        ws = torch.empty(max(lib.dsa_index_topk_workspace_bytes(T, ms, K), 4), dtype=torch.uint8, device=DEV)
        for off in (0, 1):                               # also words that start between two 8-byte lines
            got = torch.full((want.numel() + 130,), 0x5B5B5B5B, dtype=torch.int32, device=DEV)
            rc = lib.dsa_index_topk_words(p(qi), p(ki), p(wi), p(cu), T, cu.numel() - 1, Hi, Di, K, Di ** -0.5 * Hi ** -0.5, _lib.DSA_DTYPE_BF16,
                                          ms, p(got) + 4 * off, 4 * (got.numel() - off), p(ws), ws.numel(), torch.cuda.current_stream().cuda_stream)
            _lib.check(rc, "dsa_index_topk_words")
            assert torch.equal(got[off:off + want.numel()], want)
            assert bool((got[:off] == 0x5B5B5B5B).all()) and bool((got[off + want.numel():] == 0x5B5B5B5B).all())
    assert lib.dsa_index_topk_words(p(qi), p(ki), p(wi), p(cu), T, cu.numel() - 1, Hi, Di, K, 1.0, _lib.DSA_DTYPE_BF16, T, None, 0, p(ws),
                                    ws.numel(), None) == -3


@pytest.mark.parametrize("Hq,Hkv,D,segs,K,dtype", [
    (576, 144, 128, (1280, 290, 7), 16, torch.bfloat16),  # past 16 K the compacted walk, up to the last row before the gather begins
    (576, 144, 128, (1281, 290), 16, torch.bfloat16),    # and the first of the gather: the list is written after all
    (8, 2, 128, (600, 384, 290), 16, torch.bfloat16),    # too few heads for the walk: rows past 24 K gathered
    (64, 16, 128, (500, 430, 405, 400, 295), 16, torch.bfloat16),    # segments from 406 tokens on walked, shorter ones on the tiles past 24 K too: no list for this batch
    (8, 2, 128, (513, 512, 290), 16, torch.bfloat16),    # all of a segment of 32 K on the tiles, a longer one's rows past 24 K gathered
    (8, 2, 128, (500, 190, 250), 200, torch.bfloat16),   # blocks of queries that keep their whole window, also one that ends with its segment
    (4, 4, 64, (600, 41), 256, torch.bfloat16), (6, 2, 80, (500,), 127, torch.bfloat16), (4, 2, 256, (700, 64), 130, torch.bfloat16),
    (4, 1, 256, (333,), 32, torch.bfloat16), (8, 4, 48, (513, 200), 64, torch.float32), (4, 2, 128, (300,), 129, torch.float32)])
def test_attention_without_the_list(Hq, Hkv, D, segs, K, dtype):
    """The operator, with and without the list returned, against attention that was handed the list and builds its own bitmap: outputs
    and gradients bit for bit, also at crossovers that move every row to the kernels of the list or of the bitmap in the operator."""
    print("attention from words", Hq, Hkv, D, segs, K, dtype, flush=True)
    g = torch.Generator().manual_seed(D + K)
    T, cu = sum(segs), torch.tensor([0] + list(segs)).cumsum(0).int().to(DEV)
    mk = lambda *s: torch.randn(*s, generator=g).mul_(0.5).to(dtype).to(DEV)
    q, k, v, do, qi, ki, wi = mk(T, Hq, D), mk(T, Hkv, D), mk(T, Hkv, D), mk(T, Hq, D), mk(T, 4, 64), mk(T, 64), mk(T, 4)
    lib, host = _lib.load(), _lib.host()
    old, pad = lib.dsa_get_tile_crossover(), {48: 16, 80: 48}.get(D, 0)
    try:
        for crossover in (old, 0, 3):
            _lib.check(lib.dsa_set_tile_crossover(crossover), "dsa_set_tile_crossover")
            res, picked = [], None
            for listed in (True, False, None):
                a, b, c = (x.clone().requires_grad_(True) for x in (q, k, v))
                if listed is None:
                    wide = [torch.nn.functional.pad(x, (0, pad)) for x in (a, b, c)]
                    out = host.attn_node(*wide, cu, max(segs), *picked, D ** -0.5, True, False, None)[0][..., :D]
                else:
                    out = ops.dsa_varlen_attn(a, b, c, cu, max(segs), indexer_q=qi, indexer_k=ki, indexer_w=wi, top_k=K, return_indices=listed)
                if listed:
                    out, *picked = out
                out.backward(do)
                res.append((out.detach(), a.grad, b.grad, c.grad))
            for got in res[:2]:
                for x, y in zip(got, res[2]):
                    assert torch.equal(x, y)
    finally:
        lib.dsa_set_tile_crossover(old)
