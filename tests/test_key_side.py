"""The backward tile kernels (dQ; dK, dV): tile edges, pieces, operands on odd addresses; and, in the compiled code, the wait states that
their inline instructions need."""
import os
import re
import shutil
import subprocess

import pytest
import torch

from oracle import dsa_ref as R
from tests.util import assert_close_bf16
from vlm_training_amd import _lib, ops

DEV = "cuda"
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _registers(token):
    m = re.match(r"([vas])(?:\[(\d+):(\d+)\]|(\d+))$", token)
    if not m:
        return []
    lo, hi = (m.group(2), m.group(3)) if m.group(2) else (m.group(4), m.group(4))
    return [(m.group(1), r) for r in range(int(lo), int(hi) + 1)]


def _instructions(listing):
    """Functions of a listing: lists of (address, mnemonic, operands, text).  Where no address is printed, one instruction is four bytes."""
    functions, address = [[]], 0
    for line in listing.splitlines():
        text, _, note = line.partition("//")
        text = text.strip()
        if not text or text.endswith(":"):
            if text.endswith(">:"):
                functions.append([])
            continue
        op, _, rest = text.partition(" ")
        m = re.match(r"\s*([0-9A-Fa-f]+):", note)
        address = int(m.group(1), 16) if m else address + 4
        functions[-1].append((address, op, [a.strip() for a in rest.split(",")], text))
    return functions


def _scan(block, written, formed, found):
    """One basic block, entered with the wait states since registers were written by a vector instruction or formed by an MFMA on
    accumulation registers; returns them at its end."""
    clock, written, formed = 0, {r: -n for r, n in written.items()}, {r: -n for r, n in formed.items()}
    for address, op, args, text in block:
        if op == "s_nop":
            clock += int(args[0], 0) + 1
            continue
        if op.startswith("v_mfma"):
            if args[0].startswith("a["):
                if any(clock - written.get(r, -99) < 3 for a in args[1:4] for r in _registers(a)):
                    found[address] = text
                for r in _registers(args[0]):
                    formed[r] = clock
        elif op.startswith("v_"):
            if any(r[0] == "a" and clock - formed.get(r, -99) < 12 for a in args for r in _registers(a)):
                found[address] = text
            for a in args[:2 if op.startswith(("v_permlane32_swap", "v_add_co", "v_div_scale")) else 1]:
                for r in _registers(a):
                    written[r] = clock
        elif op.startswith("s_"):
            for r in _registers(args[0]):
                written.pop(r, None)
        elif op.startswith("buffer_load"):
            if any(r[0] == "s" and clock - written.get(r, -99) < 6 for a in args for r in _registers(a.split(" ")[0])):
                found[address] = text
        elif "store" in op or op.startswith("ds_write"):
            if any(r[0] == "a" and clock - formed.get(r, -99) < 12 for a in args for r in _registers(a.split(" ")[0])):
                found[address] = text
        clock += 1
    return tuple({r: clock - at for r, at in state.items() if clock - at < 12} for state in (written, formed))


def _hazards(listing):
    """(MFMAs on accumulation registers, findings).  Along every path, loops and branches followed: an operand of such an MFMA that a
    vector instruction wrote needs two wait states between them, a vector instruction or store that reads its result eleven (eight passes;
    an instruction counts as one wait state, s_nop n as n + 1).  A buffer load needs five behind a vector instruction that wrote its
    scalar operand."""
    count, found = 0, []
    for code in _instructions(listing):
        count += sum(op.startswith("v_mfma") and args[0].startswith("a[") for _, op, args, _ in code)
        at = {address: i for i, (address, *_) in enumerate(code)}
        goes = {}                                       # branches: index -> index of the target (None: outside)
        for i, (address, op, args, _) in enumerate(code):
            if op.startswith(("s_branch", "s_cbranch")):
                jump = int(args[0].split()[0], 0)
                goes[i] = at.get(address + 4 + 4 * (jump - 65536 if jump > 32767 else jump))
        ends = [i for i, (_, op, *_) in enumerate(code) if op.startswith(("s_endpgm", "s_setpc"))]
        heads = sorted({0, *(i + 1 for i in (*goes, *ends)), *(t for t in goes.values() if t is not None)} - {len(code)})
        behind = dict(zip(heads, heads[1:] + [len(code)]))
        entry, todo, bad = {h: ({}, {}) for h in heads}, list(heads) if code else [], {}
        while todo:                                     # to a fixed point: a register's wait states only fall
            h = todo.pop(0)
            out, last = _scan(code[h:behind[h]], *entry[h], bad), behind[h] - 1
            into = [goes[last]] if last in goes else []
            if last not in ends and not code[last][1].startswith("s_branch") and behind[h] < len(code):
                into.append(behind[h])
            for t in (t for t in into if t is not None):
                lower = [(mine, r, n) for mine, new in zip(entry[t], out) for r, n in new.items() if n < mine.get(r, 99)]
                for mine, r, n in lower:
                    mine[r] = n
                if lower and t not in todo:
                    todo.append(t)
        found += bad.values()
    return count, found


def test_wait_states_checker_sees_planted_hazards():
    mfma = "v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]"
    assert _hazards("v_mov_b32_e32 v3, 0\n s_nop 0\n" + mfma)[1] and not _hazards("v_mov_b32_e32 v3, 0\n s_nop 1\n" + mfma)[1]
    assert _hazards(mfma + "\n s_nop 9\n v_accvgpr_read_b32 v1, a15")[1] and not _hazards(mfma + "\n s_nop 11\n v_accvgpr_read_b32 v1, a15")[1]
    assert _hazards(mfma + "\n scratch_store_dwordx4 off, a[0:3], off")[1]
    first, load = "v_readfirstlane_b32 s5, v1\n s_nop ", "\n buffer_load_dwordx4 v2, s[4:7], 0 offen lds"
    assert _hazards(first + "3" + load)[1] and not _hazards(first + "4" + load)[1]
    # at the head of a loop, behind the last MFMA of its body (a branch counts four bytes from its own end); behind a branch around the wait
    loop = "v_accvgpr_read_b32 v1, a15\n s_nop 12\n " + mfma + "\n s_nop {}\n s_cbranch_scc1 65531\n s_endpgm"
    assert _hazards(loop.format(8))[1] and not _hazards(loop.format(9))[1]
    around = mfma + "\n s_cbranch_scc1 {}\n s_nop 11\n s_nop 0\n v_accvgpr_read_b32 v1, a15"
    assert _hazards(around.format(2))[1] and _hazards(around.format(1))[1] and not _hazards(around.format(0))[1]


def test_inline_mfmas_keep_their_wait_states(tmp_path):
    """The compiler does not see the MFMAs that these kernels issue on accumulation registers, nor their loads into LDS, so it holds none
    of their hazards back: the built library is searched for them."""
    lib = shutil.copy(_lib.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    count, kernels, found = 0, set(), []
    for name in sorted(os.listdir(tmp_path)):
        path = tmp_path / name
        held = {k for k in (b"dsa_tile_dkv_kernel", b"dsa_tile_dkv_kernel_and_dq", b"dsa_tile_dq_kernel", b"dsa_tile_fwd_kernel", b"dsa_tile_idxg_kernel", b"dsa_tile_sel_kernel",
                            b"dsa_tile_selkv_kernel") if name.endswith("gfx950") and k in path.read_bytes()}
        if held:
            kernels |= held
            c, f = _hazards(subprocess.run([OBJDUMP, "-d", str(path)], check=True, capture_output=True, text=True).stdout)
            count, found = count + c, found + f
    assert len(kernels) == 7 and count > 1000 and not found, (kernels, count, found[:5])


def _case(D, Hq, Hkv, lens, seed):
    g = torch.Generator().manual_seed(seed)
    T, cu = sum(lens), [0]
    for n in lens:
        cu.append(cu[-1] + n)
    q, k, v = (torch.randn(T, h, D, generator=g).mul_(0.5).bfloat16() for h in (Hq, Hkv, Hkv))
    return q, k, v, torch.randn(T, Hq, D, generator=g).bfloat16(), torch.tensor(cu, dtype=torch.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("D,Hq,Hkv,lens", [
    (64, 2, 2, (1, 31, 32, 33, 127, 128, 129, 257)), (64, 6, 2, (65, 2, 160, 97)), (72, 4, 4, (63, 64, 65, 190)), (96, 4, 2, (96, 33, 129)),
    (128, 3, 1, (1, 31, 33, 129, 160)), (128, 8, 8, (32, 127, 64)), (128, 16, 1, (65, 130, 5)), (128, 4, 2, (640, 3)), (256, 4, 4, (33, 128, 65)),
    (256, 16, 2, (129, 31, 64)), (256, 32, 2, (70, 300)), (256, 2, 1, (700,)),
    # enough workgroups for 64 rows or keys per wave, without and with pieces
    (64, 12, 12, (1, 31, 32, 33, 127, 128, 129, 257, 63) * 6), (72, 12, 12, (63, 64, 65, 190, 255, 256) * 7), (96, 16, 8, (96, 33, 129, 2) * 16),
    (128, 12, 4, (1, 31, 33, 129, 160) * 32), (128, 16, 16, (32, 127, 64, 193) * 12), (128, 32, 32, (700, 300, 33)), (64, 32, 32, (900, 129, 33)),
    # 64 rows and keys per wave with a causal mask too: many workgroups, or (the last two: keys, in pieces) much work
    (64, 24, 24, (1, 31, 32, 33, 127, 128, 129, 257, 63) * 6), (72, 24, 24, (63, 64, 65, 190, 255, 256) * 7), (96, 48, 24, (96, 33, 129, 2) * 16),
    (128, 48, 24, (1, 31, 33, 129, 160) * 10), (64, 128, 16, (1500, 700, 300, 33)), (128, 64, 8, (2200, 700, 129, 33))])
def test_key_and_query_gradients_at_the_edges_of_tiles(D, Hq, Hkv, lens, causal):
    print("key side", D, Hq, Hkv, lens, causal, flush=True)
    q, k, v, do, cu = _case(D, Hq, Hkv, lens, D + Hq)
    ref = [x.float().requires_grad_(True) for x in (q, k, v)]
    R.dense_varlen_causal(*ref, cu, causal=causal).backward(do.float())
    got = [x.to(DEV).requires_grad_(True) for x in (q, k, v)]
    import vlm_training_amd as M
    M.dispatch_varlen_attention(*got, cu.to(DEV), max(lens), causal=causal).backward(do.to(DEV))
    for name, a, b in zip("qkv", got, ref):
        assert_close_bf16(a.grad, b.grad, "d" + name)


@pytest.mark.gpu
@pytest.mark.parametrize("D,Hq,Hkv,lens,K", [(64, 4, 2, (200, 33), 0), (128, 6, 2, (150, 90), 40), (128, 2, 2, (700,), 0), (256, 8, 1, (129, 65), 16)])
def test_operands_on_odd_addresses_give_the_gradients(D, Hq, Hkv, lens, K):
    """The C ABI takes q and dO wherever they lie (they come through registers then)."""
    print("odd addresses", D, Hq, Hkv, lens, K, flush=True)
    q, k, v, do, cu = (x.to(DEV) for x in _case(D, Hq, Hkv, lens, 7))
    T, idx, n = q.shape[0], None, None
    if K:
        g = torch.Generator().manual_seed(1)
        idx, n = ops.index_topk(*(torch.randn(*s, generator=g).bfloat16().to(DEV) for s in ((T, 4, 64), (T, 64), (T, 4))), cu, max(lens), K)
    scale = D ** -0.5
    out, lse = ops.attn_fwd(q, k, v, idx, n, cu, max(lens), scale)

    def odd(x):
        y = torch.empty(x.numel() + 3, dtype=x.dtype, device=DEV)[3:].view_as(x)
        return y.copy_(x)

    want = ops.attn_bwd(do, q, k, v, out, lse, idx, n, cu, max(lens), scale)
    for args in ((odd(do), q), (do, odd(q)), (odd(do), odd(q))):
        got = ops.attn_bwd(*args, k, v, out, lse, idx, n, cu, max(lens), scale)
        assert torch.equal(got[0], want[0])
        # (a short launch on 16-byte boundaries runs in another form up to head_dim 128: the rounding remainder of P decided per 32 keys)
        for name, a, b in zip(("dk", "dv"), got[1:], want[1:]):
            assert_close_bf16(a, b, name)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,nseg", [(64, 1), (64, 48), (80, 48), (96, 1), (96, 48), (128, 1), (128, 48), (256, 1), (256, 48)])
def test_score_gradients_of_the_key_side_come_from_unrounded_probabilities(D, nseg, dtype):
    """Every probability is 1/96 (keys orthogonal to the queries), which bf16 rounds up by 2e-3; delta is 0 and the terms dS = P dP of a
    key all have its sign, so a rounded P would be a bias of 2e-3 in every element of dK.  What remains is rounding: of dS (2^-8 at most,
    96 independent terms per key) and of dK itself (2^-8 at most, once for the two keys of a pair): an element is off by 2^-7 at most, the
    mean over the 48 pairs of eight kv heads has a standard deviation of 2^-8 / sqrt(3 * 384) = 1.2e-4, and 8e-4 is more than six of them.
    One segment and forty-eight: 32 and, up to head_dim 128, 64 keys per wave."""
    print("unrounded P", D, nseg, dtype, flush=True)
    g = torch.Generator().manual_seed(D + nseg)
    L, H = 96, 8
    T = L * nseg
    q, k, v, do = (torch.zeros(T, H, D) for _ in range(4))
    q[..., 0] = 1.0
    v[::2, :, 1] = (1 + torch.rand(T // 2, H, generator=g)).bfloat16().float()
    v[1::2, :, 1] = -v[::2, :, 1]
    do[..., 1] = (1 + torch.rand(T, H, generator=g)).bfloat16().float()
    got = [x.to(dtype).to(DEV).requires_grad_(True) for x in (q, k, v)]
    cu = torch.arange(0, T + 1, L, dtype=torch.int32, device=DEV)
    ops.dsa_varlen_attn(*got, cu, L, softmax_scale=1.0, causal=False).backward(do.to(dtype).to(DEV))
    want = v[..., 1].double() * do[..., 1].double().view(nseg, L, H).sum(1).repeat_interleave(L, 0) / L
    ratio = got[1].grad[..., 0].double().cpu() / want - 1
    assert ratio.abs().max() <= 2.0 ** -7 and abs(ratio.mean().item()) <= 8e-4, (ratio.abs().max(), ratio.mean())
