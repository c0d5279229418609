"""Which calls of a layer take the fused form (no GPU needed): it is built for the types and sizes that `Layer` and `Runtime`
make, and everything else the op list takes or refuses must still reach the op list, not a kernel that reads its operands as
something else."""
import importlib
from types import SimpleNamespace

import numpy as np
import pytest
import torch

HOST = SimpleNamespace(float16=torch.float16, float32=torch.float32, zeros=lambda s, dtype, device: torch.zeros(s, dtype=dtype))
HEADS, HIDDEN, TOKENS = 1, 128, 5


def setup(wrq, version, tokens=TOKENS):
    mod = importlib.import_module(f"{wrq.__name__}.v{version}")
    C = 64 * HEADS
    w = mod.random_layer_weights(np.random.default_rng(version), C, HEADS, 64, HIDDEN)
    t = {k: torch.from_numpy(np.ascontiguousarray(v)) for k, v in w.items()}
    m = {k: wrq.Matrix.fp16(v) for k, v in t.items() if v.dim() >= 2}
    layer = SimpleNamespace(t={k: v for k, v in t.items() if k not in mod.QUANTIZED}, m=m)
    buf = mod.Runtime(HOST, C, HIDDEN, tokens)
    cursors = torch.zeros(tokens, dtype=torch.int32)
    return mod, layer, buf, cursors


def route(monkeypatch, mod, version, layer, buf, cursors, tokens=TOKENS, heads=HEADS, S=64, shifts=None):
    took = []
    name = {6: "dispatch_layer", 7: "dispatch_layer_ops"}[version]
    monkeypatch.setattr(mod, name, lambda *a, **k: took.append("list"))
    monkeypatch.setattr(mod, "dispatch_layer_fused", lambda *a, **k: took.append("fused"))
    state = torch.zeros((2, S + 2, heads * S))
    if version == 6:
        mod.dispatch_layer_auto(layer, buf, state, cursors, tokens, heads, S)
    else:
        getattr(mod, "dispatch_layer")(layer, buf, state, cursors, tokens, heads, S, 1, shifts=shifts)
    return took


def f32(d, *names):
    for n in names:
        (d.__setitem__(n, d[n].float()) if isinstance(d, dict) else setattr(d, n, getattr(d, n).float()))


DEVIATIONS = {
    6: {
        "f32 shift factor": lambda w, l, b: f32(l.t, "time_mix_x"),
        "f32 decay": lambda w, l, b: f32(l.t, "time_decay"),
        "f32 adapter offsets": lambda w, l, b: f32(l.t, "time_mix"),
        "f32 residual": lambda w, l, b: f32(b, "x"),
        "f32 runtime": lambda w, l, b: f32(b, "x", "att_x", "att_xx", "att_sx", "att_o", "ffn_x", "ffn_kx", "ffn_rx", "ffn_v", "ffn_r"),
        "f16 keys": lambda w, l, b: setattr(b, "att_k", b.att_k.half()),
        "packed adapter": lambda w, l, b: setattr(l.m["time_decay_w2"], "kind", "Int8"),
        "wider adapter": lambda w, l, b: l.m.__setitem__("time_mix_w1", w.Matrix.fp16(torch.zeros((320, 64), dtype=torch.float16))),
        "buffers of the op list alone": lambda w, l, b: delattr(b, "x2"),
        "buffers of fewer tokens": lambda w, l, b: setattr(b, "att_o", b.att_o[:, :3].contiguous()),
        "strided rows": lambda w, l, b: setattr(b, "x", torch.zeros((1, TOKENS, 128), dtype=torch.float16)[:, :, ::2]),
    },
    7: {
        "f32 shift factor": lambda w, l, b: f32(l.t, "x_r"),
        "f32 offsets": lambda w, l, b: f32(l.t, "w0", "a0", "v0"),
        "f32 key factor": lambda w, l, b: f32(l.t, "k_k"),
        "f32 residual": lambda w, l, b: f32(b, "x"),
        "f32 runtime": lambda w, l, b: f32(b, "x", "x2", "att_x", "att_r", "att_w", "att_n", "ffn_x"),
        "packed adapter": lambda w, l, b: setattr(l.m["g2"], "kind", "Fp4"),
        "wider adapter": lambda w, l, b: l.m.update(w1=w.Matrix.fp16(torch.zeros((96, 64), dtype=torch.float16)), w2=w.Matrix.fp16(torch.zeros((64, 96), dtype=torch.float16))),
        "first layer without v0": lambda w, l, b: l.t.pop("v0"),
        "buffers of the op list alone": lambda w, l, b: delattr(b, "x2"),
        "buffers of fewer tokens": lambda w, l, b: setattr(b, "att_n", b.att_n[:, :3].contiguous()),
        "strided rows": lambda w, l, b: setattr(b, "x", torch.zeros((1, TOKENS, 128), dtype=torch.float16)[:, :, ::2]),
    },
}


@pytest.mark.parametrize("version", [6, 7])
def test_what_layer_and_runtime_make_is_fused(wrq, monkeypatch, version):
    mod, layer, buf, cursors = setup(wrq, version)
    assert route(monkeypatch, mod, version, layer, buf, cursors) == ["fused"]
    assert route(monkeypatch, mod, version, layer, buf, torch.zeros((1, TOKENS + 3), dtype=torch.int32)) == ["fused"]


@pytest.mark.parametrize("version,what", [(v, d) for v in DEVIATIONS for d in DEVIATIONS[v]])
def test_other_types_and_sizes_take_the_op_list(wrq, monkeypatch, version, what):
    mod, layer, buf, cursors = setup(wrq, version)
    DEVIATIONS[version][what](wrq, layer, buf)
    assert route(monkeypatch, mod, version, layer, buf, cursors) == ["list"]


@pytest.mark.parametrize("version", [6, 7])
@pytest.mark.parametrize("cursors", [torch.zeros(TOKENS - 1, dtype=torch.int32), torch.zeros(2 * TOKENS, dtype=torch.int32)[::2]], ids=["too few", "strided"])
def test_cursors_that_the_op_list_refuses_reach_it(wrq, monkeypatch, version, cursors):
    mod, layer, buf, _ = setup(wrq, version)
    assert route(monkeypatch, mod, version, layer, buf, cursors) == ["list"]


@pytest.mark.parametrize("version", [6, 7])
def test_runs_beyond_the_grid_take_the_op_list(wrq, monkeypatch, version):
    A = 65536  # refused by the op list before it changes anything; the fused ops would refuse after the state was written
    mod, layer, buf, cursors = setup(wrq, version, A)
    assert route(monkeypatch, mod, version, layer, buf, cursors, A) == ["list"]


@pytest.mark.parametrize("version", [6, 7])
def test_other_heads_take_the_op_list(wrq, monkeypatch, version):
    mod, layer, buf, cursors = setup(wrq, version)
    assert route(monkeypatch, mod, version, layer, buf, cursors, heads=2, S=32) == ["list"]
    assert route(monkeypatch, mod, version, layer, buf, cursors, heads=129)[-1] == "list"


@pytest.mark.parametrize("version,names", [(6, ("time_mix_w1", "time_mix_w2", "time_decay_w1", "time_decay_w2")), (7, ("w1", "w2", "a1", "a2", "g1", "g2", "v1", "v2"))])
def test_fused_form_takes_the_adapters_of_the_matrices(wrq, monkeypatch, version, names):
    # an adapter replaced in `layer.m`, as the op list reads it, and not the tensor it was made from
    A = 20
    mod, layer, buf, cursors = setup(wrq, version, A)
    fresh = {}
    for n in names:
        fresh[n] = layer.m[n] = wrq.Matrix.fp16(torch.ones_like(layer.t[n]))
    seen = []
    for cls in ("FusedV6", "FusedV7"):
        if hasattr(mod, cls):
            recorder = type("R", (), {n: staticmethod(lambda *a, **k: seen.append(a)) for n in ("pre", "time_mix", "decay", "wkv_gate", "post_ffn", "adapters_in", "mid")})
            monkeypatch.setattr(mod, cls, recorder)
    monkeypatch.setattr(mod, "matmul_vec_group", lambda ops: None)
    monkeypatch.setattr(wrq.Matrix, "matmul_op", lambda self, *a, **k: seen.append((self.w, a)))
    monkeypatch.setattr(wrq.Matrix, "matmul_op_sparse", lambda self, *a, **k: None)
    mod.dispatch_layer_fused(layer, buf, torch.zeros((1, 66, 64)), cursors, A, 1, 64, *([1] if version == 7 else []))

    def tensors(a):
        if torch.is_tensor(a):
            yield a.data_ptr()
        elif isinstance(a, (list, tuple)):
            for e in a:
                yield from tensors(e)

    used = set(tensors(seen))
    for n in names:
        assert fresh[n].w.data_ptr() in used and layer.t[n].data_ptr() not in used, n


@pytest.mark.parametrize("C,A,tiles", [(128, 4, False), (128, 5, True), (768, 16, True), (832, 5, False), (832, 16, False), (832, 17, True), (1088, 4, False), (1088, 5, True),
                                       (2496, 5, True), (2560, 5, True), (2624, 5, False), (2624, 100, False), (2624, 225, True), (3072, 5, True), (4672, 224, False), (5120, 4, False), (5120, 5, True)])
def test_v6_adapters_of_odd_channel_counts_stay_products(wrq, C, A, tiles):
    # channels in no whole steps of 128: beyond 2560 the f16 product takes half the time of the gathered tiles in short runs
    assert importlib.import_module(f"{wrq.__name__}.v6").adapters_in_tiles(C, A) == tiles


def test_wrappers_refuse_what_the_library_cannot_see(wrq):
    h = lambda *s: torch.zeros(s, dtype=torch.float16)
    A, C, S = 4, 64, 64
    cur, state = torch.zeros(A, dtype=torch.int32), torch.zeros((1, S + 2, C))
    att, ffn = ((C, S + 1, 1), (C, S + 2, 1), (0, 0, 0)), ((C, 1, 1), (C, S + 2, 1), (0, S + 1, 0))
    x = lambda: h(A, C)
    calls = {
        "pre": lambda F, cur, v, row: F.pre(C, A, cur, x(), None, None, h(C), h(C), 1e-5, state, att, [v], x(), [row]),
        "post 6": lambda F, cur, v, row: wrq.FusedV6.post_ffn(C, A, cur, state, ffn, x(), x(), x(), x(), row, False),
        "post 7": lambda F, cur, v, row: wrq.FusedV7.post_ffn(C, A, cur, state, ffn, x(), x(), x(), row, False),
        "gate 7": lambda F, cur, v, row: wrq.FusedV7.wkv_gate(S, 1, A, cur, state, att, x(), x(), h(4, A, C), v, x(), h(C), h(C), 1e-5, row),
        "gate 6": lambda F, cur, v, row: wrq.FusedV6.wkv_gate(S, 1, A, cur, *(torch.zeros(n, C) for n in (A, 1)), state, att, *(torch.zeros(A, C) for _ in range(3)), x(),
                                                              v, h(C), 1e-5, row),
        "shift 6": lambda F, cur, v, row: wrq.FusedV6.time_mix(C, A, 32, cur, h(A, 5, 32), h(5, C, 32), h(5, C), state, att, row, h(5, A, C)),
    }
    for F in (wrq.FusedV6, wrq.FusedV7):
        for what, call in calls.items():
            for args, status in (((cur[:3], h(C), x()), wrq.ERR_SHAPE), ((cur, h(C), h(A - 1, C)), wrq.ERR_SHAPE), ((cur, h(C), x().float()), wrq.ERR_TYPE)):
                with pytest.raises(wrq.TensorError) as e:
                    call(F, *args)
                assert e.value.status == status, (what, status)
    for ops, status in (([(h(16, C), h(A, C), h(A, 8), 0)], wrq.ERR_SHAPE), ([(h(16, C), h(A, C).float(), h(A, 16), 0)], wrq.ERR_TYPE)):
        with pytest.raises(wrq.TensorError) as e:
            wrq.FusedV7.adapters_in(C, A, ops)
        assert e.value.status == status
    with pytest.raises(wrq.TensorError):
        wrq.FusedV7.pre(C, A, cur, x(), None, None, h(C), h(C), 1e-5, state, att, [h(C), h(C)], x(), [x()])
