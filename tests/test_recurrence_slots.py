"""The state recurrences where a workgroup walks one slot's tokens: more tokens than one scan of the cursors (256),
a slot that comes twice in the stack, slots without a token, a view of one slot only."""
import importlib
import os
import sys

import numpy as np
import pytest

from helpers import assert_close
from test_layer_ops import wkv6_float64, wkv6_inputs, wkv7_float64, wkv7_inputs

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
@pytest.mark.parametrize("version,S", [(5, 16), (5, 256), (6, 16), (6, 32), (6, 64), (6, 256), (7, 32), (7, 64), (7, 128)])
@pytest.mark.parametrize("B,runs", [(6, [(4, 15), (1, 241), (4, 17), (0, 3), (5, 1)]), (1, [(0, 255), (0, 18)]), (6, [(b, 1) for b in range(6)])])
def test_gpu_slots(gpu, version, S, B, runs):
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("recurrence over slots on the GPU", version, S, B, runs, flush=True)
    rng = np.random.default_rng(0x57525400 + S + B)
    H = 2
    cur = lop.pack_cursors(runs)
    A = len(cur)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    curd = dev(cur.view(np.int32))
    if version == 7:
        r, w, n, x, state = wkv7_inputs(rng, A, H, S, B, np.float32)
        sd, xd = dev(state), dev(x)
        gpu.LayerOp.time_mix_v7(curd, sd, dev(r), dev(w), dev(n), xd)
        want, want_state = wkv7_float64(cur, state, r, w, n, x)
    else:
        k, v, r, x, w, u, state = wkv6_inputs(rng, A, H, S, B, np.float32)
        if version == 5:
            w = np.broadcast_to(w[0], w.shape)
        sd, xd = dev(state), dev(x)
        (gpu.LayerOp.time_mix_v5 if version == 5 else gpu.LayerOp.time_mix_v6)(curd, dev(w[0] if version == 5 else w), dev(u), sd, dev(k), dev(v), dev(r), xd)
        want, want_state = wkv6_float64(cur, w, u, state, k, v, r, x)
    # f32 sums of S terms, the state's rounding accumulated over up to 273 tokens with a decay below 1
    assert_close(xd.cpu().numpy(), want, 5e-5, "y vs float64")
    assert_close(sd.cpu().numpy(), want_state, 5e-5, "state vs float64")


@pytest.mark.gpu
@pytest.mark.parametrize("version", [6, 7])
@pytest.mark.parametrize("runs", [[(0, 1), (1, 2), (0, 1), (0, 3), (1, 1)], [(0, 3), (0, 9), (0, 2)], [(0, 1)] * 16 + [(0, 5)]])
def test_gpu_fused_keeps_the_last_input(gpu, version, runs):
    """Requests of one slot that end close together: row 0 of the state is the layer's input at the last of them."""
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("fused recurrence, slots that come again", version, runs, flush=True)
    H, S, B = 2, 64, 2
    C = H * S
    cur = lop.pack_cursors(runs)
    A = len(cur)
    g = torch.Generator().manual_seed(0x5753 + A)
    f32 = lambda *s: (torch.randn(s, generator=g) * 0.3).cuda()
    f16 = lambda *s: f32(*s).half()
    curd, state, att_x = torch.from_numpy(cur.view(np.int32)).cuda(), f32(B, S + 2, C), f16(A, C)
    view, before = ((C, S + 1, B), (C, S + 2, B), (0, 0, 0)), att_x.clone()
    if version == 6:
        gpu.FusedV6.wkv_gate(S, H, A, curd, torch.sigmoid(f32(A, C)), f32(H, S), state, view, f32(A, C), f32(A, C), f32(A, C), f16(A, C), f16(H, S), f16(H, S),
                             64e-5, att_x)
    else:
        gpu.FusedV7.wkv_gate(S, H, A, curd, state, view, f16(A, C), f16(A, C), f16(4, A, C), f16(H, S), f16(A, C), f16(H, S), f16(H, S), 64e-5, att_x)
    slots = cur & 0xff
    for slot in set(slots.tolist()):
        last = int(np.flatnonzero(slots == slot)[-1])
        assert torch.equal(state[slot, 0], before[last].float()), slot


def column_sums(S, a, s):
    """sum_j a[j] s[j][i] in f32 as the recurrences add it: the even and the odd rows of S / 8 adjacent ones (S / 4 for S = 16) by
    fused multiply-adds, these two, then the groups in pairs, fours, ..."""
    fma = lambda x, y, z: (np.float64(x) * np.float64(y) + np.float64(z)).astype(np.float32)  # the product is exact
    groups = 8 if S >= 32 else 4
    part = np.zeros((groups, 2) + s.shape[1:], np.float32)
    for j in range(S // groups):
        rows = np.arange(groups) * (S // groups) + j
        part[:, j & 1] = fma(a[rows, None], s[rows], part[:, j & 1])
    v = part[:, 0] + part[:, 1]
    while len(v) > 1:
        v = v[0::2] + v[1::2]
    return v[0]


@pytest.mark.gpu
@pytest.mark.parametrize("A", [3, 17])  # 17: sixteen lanes per pair of columns for S = 64
@pytest.mark.parametrize("version,S", [(5, 16), (5, 64), (6, 32), (6, 64), (6, 128), (6, 256), (7, 32), (7, 64), (7, 128)])
def test_gpu_order_of_sums(gpu, version, S, A):
    """One order of the f32 sums for every form of a head size, so that results are the same bits whichever is taken."""
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("order of the recurrence's sums", version, S, A, flush=True)
    H, rng, f32 = 2, np.random.default_rng(0x57525C00 + S + A), np.float32
    fma = lambda x, y, z: (np.float64(x) * np.float64(y) + np.float64(z)).astype(f32)
    gen = lambda *s: (rng.standard_normal(s) * 0.3).astype(f32)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    k, v, r, a, kk, x, state = gen(A, H, S), gen(A, H, S), gen(A, H, S), gen(A, H, S), gen(A, H, S), gen(A, H, S), gen(1, S + 1, H * S)
    cur, sd, xd = dev(lop.pack_cursors([(0, A)]).view(np.int32)), dev(state), dev(x)
    if version == 7:
        w = np.ones((A, H, S), f32)  # the decay of an input of -200 is exp(-0)
        gpu.LayerOp.time_mix_v7(cur, sd, dev(r), dev(np.full((A, H, S), -200.0, f32)), dev(np.stack([k, v, a, kk])), xd)
    else:
        w = (1 / (1 + np.exp(-gen(A, H, S)))).astype(f32)
        w = np.broadcast_to(w[0], w.shape) if version == 5 else w
        op = gpu.LayerOp.time_mix_v5 if version == 5 else gpu.LayerOp.time_mix_v6
        op(cur, dev(w[0] if version == 5 else w), dev(np.zeros((H, S), f32)), sd, dev(k), dev(v), dev(r), xd)
    want, rows = np.empty_like(x), state[0, 1:].reshape(S, H, S).copy()
    for t in range(A):
        for h in range(H):
            s = rows[:, h]
            if version == 7:
                sa = column_sums(S, -kk[t, h], s)
                s = fma(sa, (kk[t, h] * a[t, h])[:, None], fma(s, w[t, h][:, None], k[t, h][:, None] * v[t, h]))
                want[t, h] = column_sums(S, r[t, h], s)
            else:
                want[t, h] = column_sums(S, r[t, h], s)
                s = fma(w[t, h][:, None], s, k[t, h][:, None] * v[t, h])
            rows[:, h] = s
    assert np.array_equal(xd.cpu().numpy(), want), "y"
    assert np.array_equal(sd.cpu().numpy()[0, 1:].reshape(S, H, S), rows), "state"


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [[(0, 15)], [(0, 16)], [(0, 17)], [(0, 33), (0, 7), (0, 255)], [(0, 40), (1, 1), (0, 3), (1, 20)]], ids=str)
@pytest.mark.parametrize("form", ["time_mix_v5", "time_mix_v6", "time_mix_v7", "v6 gate", "v7 gate"])
def test_gpu_wide_walk(gpu, form, runs):
    """Sixteen lanes per pair of columns where the stack has 16 tokens and more per slot: the bits that eight lanes give for
    the same stack on a state of many slots, outputs and state."""
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("wide walk of the recurrence", form, runs, flush=True)
    H, S = 3, 64
    C = H * S
    cur = lop.pack_cursors(runs)
    A, named = len(cur), 1 + max(slot for slot, _ in runs)
    curd = torch.from_numpy(cur.view(np.int32)).cuda()
    results = []
    for B in (named, 40):
        g = torch.Generator().manual_seed(0x5760 + A)
        f32 = lambda *s: (torch.randn(s, generator=g) * 0.3).cuda()
        f16 = lambda *s: f32(*s).half()
        first = f32(named, S + 1, C)
        state = torch.zeros((B, S + 1, C), device="cuda")
        state[:named] = first
        view = ((C, S + 1, B), (C, S + 1, B), (0, 0, 0))
        decay = torch.sigmoid(f32(A, H, S))
        if form == "v6 gate":
            x = f16(A, C)
            gpu.FusedV6.wkv_gate(S, H, A, curd, decay.view(A, C), f32(H, S), state, view, f32(A, C), f32(A, C), f32(A, C), f16(A, C), f16(H, S), f16(H, S), 64e-5, x)
        elif form == "v7 gate":
            x = f16(A, C)
            gpu.FusedV7.wkv_gate(S, H, A, curd, state, view, f16(A, C), f16(A, C), f16(4, A, C), f16(H, S), f16(A, C), f16(H, S), f16(H, S), 64e-5, x)
        elif form == "time_mix_v7":
            x = f16(A, H, S)
            gpu.LayerOp.time_mix_v7(curd, state, f16(A, H, S), f16(A, H, S), f16(4, A, H, S), x)
        else:
            x = f32(A, H, S)
            getattr(gpu.LayerOp, form)(curd, decay[0].contiguous() if form == "time_mix_v5" else decay, f32(H, S), state, f32(A, H, S), f32(A, H, S), f32(A, H, S), x)
        assert not state[named:].any()
        results.append((x, state[:named].clone()))
    for a, b in zip(*results):
        assert torch.isfinite(a.float()).all() and torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("op", ["channel_mix", "channel_mix_v7", "v6_post_ffn", "v7_post_ffn"])
@pytest.mark.parametrize("C", [64, 1028, 4096])
@pytest.mark.parametrize("runs", [[(0, 1)], [(0, 1), (1, 2), (0, 1), (0, 3), (1, 1)], [(1, 1)] + [(0, 1)] * 63 + [(1, 1)], [(1, 1)] * 70 + [(0, 2), (3, 1)], [(2, 255), (2, 9), (7, 3)]],
                         ids=lambda r: f"{len(r)} requests")
def test_gpu_channel_mixes_keep_the_last_input(gpu, op, C, runs):
    """The feed-forward half under the same stacks: one row of the state per slot, written from one workgroup per token."""
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("channel mix, slots that come again", op, C, runs[:6], flush=True)
    B = 4  # a slot beyond the state counts as the last one
    cur = lop.pack_cursors(runs)
    A = len(cur)
    g = torch.Generator().manual_seed(0x5758 + A + C)
    f16 = lambda *s: torch.randn(s, generator=g).half().cuda()
    curd, state, view = torch.from_numpy(cur.view(np.int32)).cuda(), torch.randn((B, 1, C), generator=g).cuda(), ((C, 1, B), (C, 1, B), (0, 0, 0))
    r, v, x, x_in, out = (f16(1, A, C) for _ in range(5))
    want, rows = state.clone(), x.clone()
    for t in range(A):
        slot, first, n = int(cur[t]) & 0xff, int(cur[t]) >> 8 & 0xffff, int(cur[t]) >> 24
        if t - first + 1 == n:
            want[min(slot, B - 1), 0] = rows[0, t].float()
    if op == "channel_mix":
        gpu.LayerOp.channel_mix(curd, state, r, v, x)
    elif op == "channel_mix_v7":
        gpu.LayerOp.channel_mix_v7(curd, state, v, x)
    elif op == "v6_post_ffn":
        gpu.FusedV6.post_ffn(C, A, curd, state, view, r, v, x, x_in, out, False)
    else:
        gpu.FusedV7.post_ffn(C, A, curd, state, view, v, x, x_in, out, False)
    assert torch.equal(state, want)


@pytest.mark.gpu
@pytest.mark.parametrize("B,runs", [(2, [(1, 1)]), (300, [(255, 1)]), (9, [(3, 2), (0, 1), (3, 1)]), (9, [(9, 1), (2, 3), (8, 2)]), (300, [(255, 2), (0, 1), (254, 9), (255, 1)]),
                                    (256, [(i, 1) for i in range(200, 0, -1)] + [(77, 54)]), (256, [(5, 255)])], ids=lambda v: str(v if isinstance(v, int) else len(v)))
@pytest.mark.parametrize("form", ["time_mix_v5", "time_mix_v6", "time_mix_v7", "v6 gate", "v7 gate"])
def test_gpu_more_slots_than_tokens(gpu, form, B, runs):
    """A state of more slots than the run has tokens gives what a state of the named slots alone gives, bit for bit, and
    leaves the other slots as they are."""
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("more slots than tokens", form, B, runs[:4], flush=True)
    H, S = 2, 64
    C = H * S
    named = sorted({min(slot, B - 1) for slot, _ in runs})
    few = [(named.index(min(slot, B - 1)), n) for slot, n in runs]
    A = sum(n for _, n in runs)
    g = torch.Generator().manual_seed(0x575A + A)
    f32 = lambda *s: (torch.randn(s, generator=g) * 0.3).cuda()
    f16 = lambda *s: f32(*s).half()
    state, x0 = f32(B, S + 2, C), (f16 if "gate" in form else f32)(A, H, S)
    k, v, r, u, decay, kvak = f32(A, H, S), f32(A, H, S), f32(A, H, S), f32(H, S), torch.sigmoid(f32(A, H, S)), f32(4, A, H, S)
    gates, gw, gb = f16(A, C), f16(H, S), f16(H, S)
    outs = []
    for stack, rows in ((runs, state.clone()), (few, state[named].contiguous())):
        n = rows.shape[0]
        cur, x, view = torch.from_numpy(lop.pack_cursors(stack).view(np.int32)).cuda(), x0.clone(), ((C, S + 1, n), (C, S + 2, n), (0, 0, 0))
        if form == "time_mix_v7":
            gpu.LayerOp.time_mix_v7(cur, rows, r, k, kvak, x, state_view=view)
        elif form == "v6 gate":
            gpu.FusedV6.wkv_gate(S, H, A, cur, decay, u, rows, view, k, v, r, gates, gw, gb, 64e-5, x)
        elif form == "v7 gate":
            gpu.FusedV7.wkv_gate(S, H, A, cur, rows, view, r.half(), k.half(), kvak.half(), gw, gates, gw, gb, 64e-5, x)
        else:
            getattr(gpu.LayerOp, form)(cur, decay[0].contiguous() if form == "time_mix_v5" else decay, u, rows, k, v, r, x, state_view=view)
        outs.append((x, rows))
    assert torch.equal(outs[0][0], outs[1][0])
    want = state.clone()
    want[named] = outs[1][1]
    assert torch.equal(outs[0][1], want)


@pytest.mark.gpu
@pytest.mark.parametrize("version", [6, 7])
@pytest.mark.parametrize("B,runs", [(6, [(4, 15), (1, 241), (4, 17), (0, 3), (5, 1)]), (2, [(0, 250), (1, 2), (0, 20), (1, 255), (0, 9)]), (1, [(0, 255), (0, 255), (0, 3)])])
def test_gpu_fused_beyond_one_scan_of_the_cursors(gpu, version, B, runs):
    """The gate forms over more tokens than one scan of the cursors (256), a slot that comes again behind the edge and a
    single one: output and whole state against the op list (recurrence, group norm, gate) on the same operands."""
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("gate forms beyond one scan", version, B, runs, flush=True)
    H, S = 2, 64
    C, cur = H * S, lop.pack_cursors(runs)
    A = len(cur)
    g = torch.Generator().manual_seed(0x575B + A)
    f32 = lambda *s: (torch.randn(s, generator=g) * 0.3).cuda()
    f16 = lambda *s: f32(*s).half()
    curd, view = torch.from_numpy(cur.view(np.int32)).cuda(), ((C, S + 1, B), (C, S + 2, B), (0, 0, 0))
    state, x, gate, gw, gb = f32(B, S + 2, C), f16(A, H, S), f16(A, H, S), f16(H, S), f16(H, S)
    want, y = state.clone(), None
    if version == 6:
        k, v, r, u, w = f32(A, H, S), f32(A, H, S), f32(A, H, S), f32(H, S), torch.sigmoid(f32(A, H, S))
        y = x.float()
        gpu.LayerOp.time_mix_v6(curd, w, u, want, k, v, r, y, state_view=view)
        gpu.LayerOp.group_norm(gw, gb, y, 64e-5)
        y = y.half()
        gpu.LayerOp.mul_activate(gate, y, gpu.ACT_SILU)
        gpu.FusedV6.wkv_gate(S, H, A, curd, w, u, state, view, k, v, r, gate, gw, gb, 64e-5, x)
    else:
        r, w, n, u = f16(A, H, S), f16(A, H, S), f16(4, A, H, S), f16(H, S)
        y = x.clone()
        gpu.LayerOp.time_mix_v7(curd, want, r, w, n, y, state_view=view)
        gpu.LayerOp.group_norm(gw, gb, y, 64e-5)
        gpu.LayerOp.time_first_v7(u, r, n, y)
        gpu.LayerOp.mul(gate, y)
        gpu.FusedV7.wkv_gate(S, H, A, curd, state, view, r, w, n, u, gate, gw, gb, 64e-5, x)
    # the same roundings to f16 on both sides; f32 sums in another order flip one here and there: an ulp (2^-10) of values up to 4
    assert_close(x.cpu().numpy(), y.cpu().numpy(), 4e-3, "gated output")
    assert_close(state.cpu().numpy(), want.cpu().numpy(), 1e-6, "state")
