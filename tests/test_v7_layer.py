"""Two consecutive RWKV-v7 layers (the first keeps its values as `v0`, the second mixes its own with
them), fused and op by op like the reference (src/runtime/v7.rs:704-1006), on the GPU through the
library against a numpy composition of the oracle's restatements."""
import importlib
import os
import sys

import numpy as np
import pytest

from helpers import assert_close, int8_dequant64, nf4_dequant64

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SEED = 0x57525700


def layer_numpy(lop, w, x, v0, state, cursors, H, S, index):
    """The layer on the CPU, every buffer rounded to f16 as the reference's runtime keeps it
    (src/runtime/v7.rs:281-320).  Returns the new x and the values the first layer hands on."""
    f16, f64 = np.float16, np.float64
    A, C = x.shape
    mm = lambda a, W: (a.astype(f64) @ W.astype(f64).T)
    att_x = lop.layer_norm(w["att_ln_w"], w["att_ln_b"], x, 1e-5)
    rx, wx, kx, vx, ax, gx = (lop.token_shift(cursors, w[n], state[:, 0], att_x, f16, reversed=True)[0] for n in ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g"))
    r, k, v = mm(rx, w["att_w_r"]).astype(f16), mm(kx, w["att_w_k"]).astype(f16), mm(vx, w["att_w_v"]).astype(f16)
    aux_w = np.tanh(mm(wx, w["w1"])).astype(f16)
    att_w = lop.binary("add", w["w0"], mm(aux_w, w["w2"]).astype(f16))
    aux_a = mm(ax, w["a1"]).astype(f16)
    att_a = lop.binary("add", w["a0"], mm(aux_a, w["a2"]).astype(f16), act_out=6)
    aux_g = lop.activation(6, mm(gx, w["g1"]).astype(np.float32)).astype(f16)
    att_g = mm(aux_g, w["g2"]).astype(f16)
    kk = lop.binary("mul", w["k_k"], k)
    kk = lop.l2_norm(kk.reshape(A, H, S), 1e-12).reshape(A, C)
    k = lop.control_k_v7(w["k_a"], att_a, k)
    if index == 0:
        v0 = v.copy()
    else:
        aux_v = mm(vx, w["v1"]).astype(f16)
        vv = lop.binary("add", w["v0"], mm(aux_v, w["v2"]).astype(f16), act_out=6)
        v = lop.lerp(v0, v, vv, reversed=True)
    n = np.stack([k, v, att_a, kk]).reshape(4, A, H, S)
    att = np.ascontiguousarray(state[:, :S + 1])
    y = lop.time_mix_v7(cursors, att, r.reshape(A, H, S), att_w.reshape(A, H, S), n, att_x.reshape(A, H, S))
    state[:, :S + 1] = att
    y = lop.group_norm(w["gn_w"], w["gn_b"], y, 64e-5)
    y = lop.time_first_v7(w["r_k"], r.reshape(A, H, S), n, y)
    att_x = lop.binary("mul", att_g, y.reshape(A, C))
    x = lop.binary("add", mm(att_x, w["att_w_o"]).astype(f16), x)
    ffn_x = lop.layer_norm(w["ffn_ln_w"], w["ffn_ln_b"], x, 1e-5)
    ffn_state = np.ascontiguousarray(state[:, S + 1])
    fkx = lop.token_shift(cursors, w["ffn_x_k"], ffn_state, ffn_x, f16, reversed=True)[0]
    fk = lop.activation(1, mm(fkx, w["ffn_w_k"]).astype(np.float32)).astype(f16)
    fv = mm(fk, w["ffn_w_v"]).astype(f16)
    ffn_x = lop.channel_mix_v7(cursors, ffn_state, fv, ffn_x)
    state[:, S + 1] = ffn_state
    return lop.binary("add", ffn_x, x), v0


@pytest.mark.gpu
@pytest.mark.parametrize("quant", ["int8", "nf4"])
@pytest.mark.parametrize("runs", [[(2, 3), (0, 1), (5, 4)], [(1, 20), (3, 12)], [(4, 1)]], ids=["8 tokens", "32 tokens (chunk kernels)", "1 token"])
@pytest.mark.parametrize("form", ["dispatch_layer", "dispatch_layer_ops"])
def test_v7_layers_against_numpy(gpu, oracle, quant, runs, form):
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    v7 = importlib.import_module(gpu.__name__ + ".v7")
    print("v7 layers on the GPU", quant, runs, flush=True)
    H, S, hidden, B, L = 4, 64, 1024, 6, 2
    C = H * S
    rng = np.random.default_rng(SEED + len(runs))
    cursors = lop.pack_cursors(runs)
    A = len(cursors)
    x = rng.standard_normal((A, C)).astype(np.float16)
    curd = torch.from_numpy(cursors.view(np.int32)).cuda()
    buf = v7.Runtime(torch, C, hidden, A)
    buf.x.copy_(torch.from_numpy(x).cuda().reshape(1, A, C))
    want, v0 = x, None
    for index in range(L):
        w = v7.random_layer_weights(rng, C, H, S, hidden)
        state = (0.1 * rng.standard_normal((B, S + 2, C))).astype(np.float32)
        layer = v7.Layer(torch, w, quant)
        wq = dict(w)  # the CPU side works on what the packed matrices represent
        for name in v7.QUANTIZED:
            mtx = layer.m[name]
            if quant == "int8":
                wq[name] = int8_dequant64(mtx.w.cpu().numpy(), mtx.m.cpu().numpy())
            else:
                wq[name] = nf4_dequant64(mtx.w.cpu().numpy(), mtx.m.cpu().numpy(), np.array(gpu.NF4_QUANT, dtype=np.float32))
        want_state = state.copy()
        want, v0 = layer_numpy(lop, wq, want, v0, want_state, cursors, H, S, index)
        sd = torch.from_numpy(state.copy()).cuda()
        assert v7.fused_is_built(layer, H, S, buf, curd, A)  # which dispatch_layer then takes
        getattr(v7, form)(layer, buf, sd, curd, A, H, S, index)
        torch.cuda.synchronize()
        got = buf.x.cpu().numpy()[0]
        # f16 buffers between 50 ops: a few f16 ulps of the O(1) activations
        assert_close(got, want, 1.5e-2, f"output of layer {index}")
        assert_close(sd.cpu().numpy(), want_state, 1.5e-2, f"state of layer {index} after the run")
        untouched = [b for b in range(B) if b not in [s for s, _ in runs]]
        assert np.array_equal(sd.cpu().numpy()[untouched], state[untouched])
        want = got  # the next layer starts from the device's x on both sides


@pytest.mark.gpu
@pytest.mark.parametrize("runs", [[(2, 3), (0, 1), (5, 4)], [(1, 32)], [(4, 1)]], ids=["8 tokens", "32 tokens", "1 token"])
def test_v7_layer_packed_token_shifts_equal_the_op_list(gpu, runs):
    # the six token shifts in one launch (factors stacked and repeated over the tokens with `broadcast`): bit-equal
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    v7 = importlib.import_module(gpu.__name__ + ".v7")
    print("v7 layer, packed token shifts", runs, flush=True)
    H, S, hidden, B = 4, 64, 1024, 6
    C = H * S
    rng = np.random.default_rng(SEED + 50 + len(runs))
    cursors = lop.pack_cursors(runs)
    A = len(cursors)
    curd = torch.from_numpy(cursors.view(np.int32)).cuda()
    layer = v7.Layer(torch, v7.random_layer_weights(rng, C, H, S, hidden), "int8")
    x = rng.standard_normal((A, C)).astype(np.float16)
    state = (0.1 * rng.standard_normal((B, S + 2, C))).astype(np.float32)
    outs = []
    for packed in (False, True):
        buf = v7.Runtime(torch, C, hidden, A)
        buf.x.copy_(torch.from_numpy(x).cuda().reshape(1, A, C))
        buf.att_v0.copy_(torch.from_numpy(x[::-1].copy()).cuda().reshape(1, A, C))
        sd = torch.from_numpy(state.copy()).cuda()
        v7.dispatch_layer_ops(layer, buf, sd, curd, A, H, S, 1, shifts=v7.PackedShifts(torch, layer, A) if packed else None)
        torch.cuda.synchronize()
        outs.append((buf.x.cpu().numpy(), sd.cpu().numpy()))
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])


@pytest.mark.gpu
@pytest.mark.parametrize("H", [1, 17, 33, 65], ids=lambda h: f"{64 * h} channels")
@pytest.mark.parametrize("runs", [[(4, 1)], [(2, 3), (0, 12), (5, 1)], [(1, 15), (3, 2)], [(i, 1) for i in range(5)] + [(5, 251)]],
                         ids=["1 token", "16 tokens", "17 tokens", "256 tokens"])
def test_v7_layer_fused_equals_op_list(gpu, runs, H):
    # edges of the fused kernels: one row vector per thread up to eight (channels), whole and ragged tiles of 16 tokens,
    # the first layer (no adapter v) and a later one.  The bound is the v6 layer's: both sides round the same f16
    # buffers, sums in another order move single values by an ulp (2^-11) and the products behind carry a few of them on
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    v7 = importlib.import_module(gpu.__name__ + ".v7")
    print("v7 layer, fused", runs, H, flush=True)
    S, hidden, B = 64, 256, 6
    C = H * S
    rng = np.random.default_rng(SEED + 90 + len(runs) + H)
    cursors = lop.pack_cursors(runs)
    A = len(cursors)
    curd = torch.from_numpy(cursors.view(np.int32)).cuda()
    layer = v7.Layer(torch, v7.random_layer_weights(rng, C, H, S, hidden), "int8" if C % 128 == 0 or H > 1 else "nf4")
    assert v7.fused_is_built(layer, H, S)
    x, v0 = (rng.standard_normal((1, A, C)).astype(np.float16) for _ in range(2))
    state = (0.1 * rng.standard_normal((B, S + 2, C))).astype(np.float32)
    for index, rescale in ((0, False), (1, True)):
        outs = []
        for dispatch in (v7.dispatch_layer_ops, v7.dispatch_layer_fused):
            buf = v7.Runtime(torch, C, hidden, A)
            buf.x.copy_(torch.from_numpy(x).cuda())
            buf.att_v0.copy_(torch.from_numpy(v0).cuda())
            sd = torch.from_numpy(state.copy()).cuda()
            dispatch(layer, buf, sd, curd, A, H, S, index, rescale)
            torch.cuda.synchronize()
            outs.append((buf.x.cpu().numpy(), sd.cpu().numpy(), buf.att_v0.cpu().numpy()))
        for i, what in enumerate(("layer output", "state", "first layer's values")):
            assert_close(outs[1][i], outs[0][i], 4e-3, f"{what}, fused vs op list")


@pytest.mark.gpu
@pytest.mark.parametrize("packed", [False, True], ids=["six shifts", "packed shifts"])
@pytest.mark.parametrize("runs", [[(4, 1)], [(2, 3), (0, 13), (5, 1)], [(1, 20), (3, 13)]], ids=["1 token", "17 tokens", "33 tokens"])
def test_v7_dispatch_leaves_the_buffers_of_the_op_list(gpu, runs, packed):
    # every buffer of the run, not the layer's output alone: a caller may read any of them behind `dispatch_layer`.
    # The bound is that of the fused layer against the op list above
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    v7 = importlib.import_module(gpu.__name__ + ".v7")
    print("v7 layer, buffers", runs, packed, flush=True)
    H, S, hidden, B = 3, 64, 256, 6
    C = H * S
    rng = np.random.default_rng(SEED + 130 + len(runs))
    cursors = lop.pack_cursors(runs)
    A = len(cursors)
    curd = torch.from_numpy(cursors.view(np.int32)).cuda()
    layer = v7.Layer(torch, v7.random_layer_weights(rng, C, H, S, hidden), "int8")
    x, v0 = (rng.standard_normal((1, A, C)).astype(np.float16) for _ in range(2))
    state = (0.1 * rng.standard_normal((B, S + 2, C))).astype(np.float32)
    for index in (0, 1):
        outs = []
        for dispatch in (v7.dispatch_layer_ops, v7.dispatch_layer):
            buf = v7.Runtime(torch, C, hidden, A)
            assert v7.fused_is_built(layer, H, S, buf, curd, A)
            buf.x.copy_(torch.from_numpy(x).cuda())
            buf.att_v0.copy_(torch.from_numpy(v0).cuda())
            shifts = v7.PackedShifts(torch, layer, A) if packed else None
            dispatch(layer, buf, torch.from_numpy(state.copy()).cuda(), curd, A, H, S, index, shifts=shifts)
            torch.cuda.synchronize()
            named = {name: t for name, t in vars(buf).items() if name != "x2"}
            if packed:
                named["sx"] = shifts.sx
            outs.append({name: t.cpu().numpy() for name, t in named.items()})
        for name in outs[0]:
            assert_close(outs[1][name], outs[0][name], 4e-3, f"{name} of layer {index}")


@pytest.mark.gpu
def test_v7_dispatch_takes_the_factors_of_packed_shifts(gpu):
    # factors of its own in `PackedShifts.mix`, another for every token, as the op list takes them; the bound as above
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    v7 = importlib.import_module(gpu.__name__ + ".v7")
    H, S, hidden, B = 2, 64, 256, 4
    C = H * S
    rng = np.random.default_rng(SEED + 140)
    cursors = lop.pack_cursors([(1, 5), (3, 1), (0, 12)])
    A = len(cursors)
    curd = torch.from_numpy(cursors.view(np.int32)).cuda()
    layer = v7.Layer(torch, v7.random_layer_weights(rng, C, H, S, hidden), "int8")
    x, mix = rng.standard_normal((1, A, C)).astype(np.float16), rng.random((6, A, C)).astype(np.float16)
    state = (0.1 * rng.standard_normal((B, S + 2, C))).astype(np.float32)
    outs = []
    for dispatch in (v7.dispatch_layer_ops, v7.dispatch_layer):
        buf, shifts = v7.Runtime(torch, C, hidden, A), v7.PackedShifts(torch, layer, A)
        shifts.mix.copy_(torch.from_numpy(mix).cuda())
        assert v7.fused_is_built(layer, H, S, buf, curd, A, shifts)
        buf.x.copy_(torch.from_numpy(x).cuda())
        sd = torch.from_numpy(state.copy()).cuda()
        dispatch(layer, buf, sd, curd, A, H, S, 0, shifts=shifts)
        torch.cuda.synchronize()
        outs.append([t.cpu().numpy() for t in (shifts.sx, buf.x, sd)])
    for i, what in enumerate(("shifted rows", "layer output", "state")):
        assert_close(outs[1][i], outs[0][i], 4e-3, what)


@pytest.mark.gpu
def test_v7_mid_of_the_first_layer_needs_no_adapter_v(gpu):
    import torch

    S, H, A = 64, 2, 17
    C = S * H
    g = torch.Generator().manual_seed(SEED + 150)
    h = lambda *s: (0.3 * torch.randn(s, generator=g)).half().cuda()
    aux, w2, vectors = [h(A, r) for r in (64, 64, 128, 32)], [h(C, r) for r in (64, 64, 128, 32)], [h(C) for _ in range(5)]
    k, v = h(A, C), h(A, C)
    outs = []
    for last in (None, 0):
        x, w, b = (list(a) for a in (aux, w2, vectors))
        if last is None:
            x[3], w[3], b[2] = None, None, None
        out = [torch.empty((A, C), dtype=torch.float16, device="cuda") for _ in range(3)] + [torch.empty((4, A, C), dtype=torch.float16, device="cuda")]
        gpu.FusedV7.mid(S, H, A, True, x, w, b, 1e-12, k, v, *out)
        outs.append(out)
    for a, b in zip(*outs):
        assert torch.equal(a, b)
    assert torch.equal(outs[0][0], v) and torch.equal(outs[0][3][1], v)


@pytest.mark.gpu
@pytest.mark.parametrize("H", [1, 17, 65], ids=lambda h: f"{64 * h} channels")
@pytest.mark.parametrize("B,runs", [(6, [(1, 9), (0, 230), (4, 14), (2, 41), (5, 2)]), (1, [(0, 255), (0, 45)])], ids=["slots", "one slot"])
def test_v7_layer_fused_beyond_one_scan_of_the_cursors(gpu, B, runs, H):
    # runs of more than 256 tokens, the fused layer against the op list.  Either side is 7e-4 of the norm away from 64 bits
    # (roundings of the f16 buffers), so they differ by up to 1e-3 of it; of 1.2 million values of rms 1.2 the largest
    # difference is then 4.9 sigma = 6e-3
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    v7 = importlib.import_module(gpu.__name__ + ".v7")
    print("v7 layer beyond 256 tokens", runs, H, flush=True)
    S, hidden = 64, 256
    C = H * S
    rng = np.random.default_rng(SEED + 160 + H)
    cursors = lop.pack_cursors(runs)
    A = len(cursors)
    curd = torch.from_numpy(cursors.view(np.int32)).cuda()
    layer = v7.Layer(torch, v7.random_layer_weights(rng, C, H, S, hidden), "int8")
    x, v0 = (rng.standard_normal((1, A, C)).astype(np.float16) for _ in range(2))
    state = (0.1 * rng.standard_normal((B, S + 2, C))).astype(np.float32)
    outs = []
    for dispatch in (v7.dispatch_layer_ops, v7.dispatch_layer):
        buf = v7.Runtime(torch, C, hidden, A)
        assert v7.fused_is_built(layer, H, S, buf, curd, A)
        buf.x.copy_(torch.from_numpy(x).cuda())
        buf.att_v0.copy_(torch.from_numpy(v0).cuda())
        sd = torch.from_numpy(state.copy()).cuda()
        dispatch(layer, buf, sd, curd, A, H, S, 1)
        torch.cuda.synchronize()
        outs.append((buf.x.cpu().numpy().astype(np.float64), sd.cpu().numpy().astype(np.float64)))
    for i, what in enumerate(("layer output", "state")):
        assert_close(outs[1][i], outs[0][i], 8e-3, what)
        assert np.linalg.norm(outs[1][i] - outs[0][i]) < 1.5e-3 * np.linalg.norm(outs[0][i]), what
