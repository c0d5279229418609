"""CPU-side checks of the C ABI: the library loads, exports what include/wrq.h declares,
and rejects bad operands before touching a device (no compute calls here)."""
import ctypes as C
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def declared_functions():
    text = open(os.path.join(ROOT, "include", "wrq.h")).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(wrq_[a-z0-9_]+)\s*\(", text)))


def test_library_exports_every_declared_symbol(wrq):
    L = wrq.lib()
    names = declared_functions()
    assert set(wrq.EXPORTS) == set(names)
    for n in names:
        assert hasattr(L, n), n
    assert L.wrq_abi_version() == 1
    assert L.wrq_abi_minor() >= 3  # entry points were added since minor 0; signatures never changed
    assert L.wrq_status_string(0) == b"ok"
    assert L.wrq_status_string(1) == b"tensor shape not match"


def test_struct_layouts_match_the_header(wrq):
    # wrq_view is the reference's 48-byte View uniform (src/tensor/mod.rs:26-43)
    assert C.sizeof(wrq.CView) == 48
    assert C.sizeof(wrq.CTensor) == 24
    assert C.sizeof(wrq.CTensorView) == 8 + 48 + 8
    assert wrq.ACTIVATIONS[1] == "squared_relu" and len(wrq.ACTIVATIONS) == 8


@pytest.mark.parametrize("shape", [(64,), (3, 64), (2, 3, 64), (5, 2, 3, 64), (0, 64)], ids=str)
def test_packed_descriptors_equal_the_structures(wrq, shape):
    import torch

    for dtype in (torch.float16, torch.float32, torch.uint8):
        t = torch.zeros(shape, dtype=dtype)
        assert wrq._tensor(t) == bytes(wrq.as_tensor(t))
        assert wrq._view(t) == bytes(wrq.as_view(t)) and wrq._view(t, dtype=wrq.F16) == bytes(wrq.as_view(t, dtype=wrq.F16))
    for view in (((64, 1, 1), (64, 3, 2), (0, 2, 1)), ([32, 2], [64, 3], [16, 1]), ((4, 1, 1, 1), (64, 3, 2, 5), (0, 0, 0, 4)), ((), (), ())):
        assert wrq._view(t, view) == bytes(wrq.as_view(t, view))


def test_packed_descriptors_leave_odd_values_to_the_structures(wrq):
    import torch

    t = torch.zeros((2, 64))
    for view in (((64, 2 ** 32 + 1), (64, 2), (0, 0)), ((64, 2), (64, 2), (-4, 0))):  # wrapped to 32 bits, for the library to judge
        assert bytes(wrq._view(t, view)._obj) == bytes(wrq.as_view(t, view))
    for bad in (((64.5, 2), (64, 2), (0, 0)), ((1,) * 5, (64, 2), (0, 0))):
        with pytest.raises((TypeError, IndexError, ValueError, RuntimeError)):
            wrq.as_view(t, bad)
        with pytest.raises((TypeError, IndexError, ValueError, RuntimeError)):
            wrq._view(t, bad)
    for make in (wrq._tensor, wrq._view):
        with pytest.raises(AssertionError):
            make(t.t())


FAKE = 0x10000  # never dereferenced: every call below fails its checks first


def T(wrq, shape, ptr=FAKE):
    return wrq.CTensor(ptr, tuple(shape))


def V(wrq, shape, stride=None, offset=(0, 0, 0, 0), dtype=0, ptr=FAKE):
    return wrq.CTensorView(ptr, wrq.CView(tuple(shape), tuple(stride or shape), tuple(offset)), dtype)


def err(wrq):
    return wrq.lib().wrq_last_error().decode()


def test_binding_tells_tensors_from_views(wrq):
    L = wrq.lib()
    t, v = T(wrq, (64, 1, 1, 1)), V(wrq, (64, 1, 1, 1))
    for tensor in (t, C.byref(t), C.pointer(t)):  # a structure goes by itself, by reference or by pointer
        assert L.wrq_softmax(None, tensor, 7) == wrq.ERR_TYPE
    for view in (v, C.byref(v), C.pointer(v)):
        assert L.wrq_activate(None, view, 99) == wrq.ERR_UNSUPPORTED
    assert L.wrq_softmax(None, None, 0) == wrq.ERR_NULL
    for other in (v, C.byref(v), C.pointer(v), FAKE, bytes(v), bytes(8)):
        with pytest.raises(C.ArgumentError):
            L.wrq_softmax(None, other, 7)
    for other in (t, C.byref(t), C.pointer(t), FAKE, bytes(t), bytes(8)):
        with pytest.raises(C.ArgumentError):
            L.wrq_activate(None, other, 99)


def test_wrappers_hand_over_the_descriptors_declared(wrq, monkeypatch):
    """Every wrapper against the argument types of its entry point: a tensor's bytes where a tensor is read, a view's where a view is."""
    import inspect

    import torch

    sizes = {C.POINTER(wrq.CTensor): C.sizeof(wrq.CTensor), C.POINTER(wrq.CTensorView): C.sizeof(wrq.CTensorView)}
    typed, seen = wrq.lib(), {}

    class Recorder:
        def __getattr__(self, name):
            def call(*args):
                want = getattr(typed, name).argtypes
                assert len(args) == len(want), name
                for k, (arg, kind) in enumerate(zip(args, want)):
                    if kind in sizes:
                        assert type(arg) is bytes and len(arg) == sizes[kind], (name, k)
                    else:
                        assert type(arg) is not bytes, (name, k)
                seen[name] = seen.get(name, 0) + 1
                return wrq.OK

            return call

    monkeypatch.setattr(wrq, "_packed", Recorder)
    monkeypatch.setattr(wrq, "_stream", lambda: 0)
    t = torch.zeros((2, 64), dtype=torch.float16)
    view = ((64, 2), (64, 2), (0, 0))
    plain = dict(eps=1e-5, scale=1.0, bias=0.0, act=0, act_x=0, act_y=0, act_out=0, sparse=False, reversed=False, rescale=False, first=False, checked=True,
                 Cn=64, S=64, H=1, A=2, lora_size=32, factors=[t], shifts=[t], aux=[t] * 4, vectors=[t] * 5, buffers=[None] * 5, ops=[(t, t, t, 0)])
    for cls in (wrq.TensorOp, wrq.LayerOp, wrq.FusedV6, wrq.FusedV7):
        for name, f in vars(cls).items():
            if not isinstance(f, staticmethod) or name.startswith("_"):
                continue
            names = list(inspect.signature(f.__func__).parameters)
            plain["w2"] = [t] * 4 if "aux" in names else t
            for views in (None, view):
                f.__func__(**{n: views if n == "view" or n.endswith("_view") else plain.get(n, t) for n in names})
    described = {n for n in wrq.EXPORTS if any(a in sizes for a in getattr(typed, n).argtypes or ())}
    older = {"wrq_v7_post_ffn"}  # the wrapper calls its _buffers form
    assert described - older <= set(seen), described - older - set(seen)


def test_shape_errors_read_like_the_reference(wrq):
    L = wrq.lib()
    K, R, Tn = 256, 8, 1
    ok_mm = T(wrq, (2 * K * R // 128, 1, 1, 1))
    # minmax of the wrong length -> TensorErrorKind::Shape(got, want) (src/tensor/ops.rs:809)
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(T(wrq, (7, 1, 1, 1))),
                              C.byref(V(wrq, (K, Tn, 1, 1))), C.byref(V(wrq, (R, Tn, 1, 1))), 0, 0)
    assert s == wrq.ERR_SHAPE
    assert err(wrq) == "tensor shape not match: (7, 1, 1, 1) vs. (32, 1, 1, 1)"
    # matrix vs input K mismatch (ops.rs:810)
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(ok_mm),
                              C.byref(V(wrq, (K // 2, Tn, 1, 1))), C.byref(V(wrq, (R, Tn, 1, 1))), 0, 0)
    assert s == wrq.ERR_SHAPE and "(256, 8, 1, 1) vs. (128, 8, 1, 1)" in err(wrq)
    # token count mismatch between input and output (ops.rs:811)
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(ok_mm),
                              C.byref(V(wrq, (K, 2, 1, 1))), C.byref(V(wrq, (R, 1, 1, 1))), 0, 0)
    assert s == wrq.ERR_SHAPE and "(256, 2, 1, 1) vs. (256, 1, 1, 1)" in err(wrq)
    # nf4: matrix holds K/2 bytes per row, absmax one per 64 (ops.rs:910-912)
    s = L.wrq_matmul_vec_nf4(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(T(wrq, (16, 1, 1, 1))),
                             C.byref(T(wrq, (K * R // 64, 1, 1, 1))), C.byref(V(wrq, (K, Tn, 1, 1))),
                             C.byref(V(wrq, (R, Tn, 1, 1))), 0, 0)
    assert s == wrq.ERR_SHAPE
    # quantize: input and output shapes must agree (ops.rs:2405), minmax = 2 * ceil(len / 128) (ops.rs:2402-2403)
    s = L.wrq_quantize_mat_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(ok_mm), C.byref(T(wrq, (K, R + 4, 1, 1))))
    assert s == wrq.ERR_SHAPE
    s = L.wrq_quantize_mat_nf4(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(T(wrq, (16, 1, 1, 1))),
                               C.byref(T(wrq, (K * R // 64 + 1, 1, 1, 1))), C.byref(T(wrq, (K // 2, R, 1, 1))))
    assert s == wrq.ERR_SHAPE and "(33, 1, 1, 1) vs. (32, 1, 1, 1)" in err(wrq)


def test_unchecked_preconditions_of_the_reference_become_errors(wrq):
    L = wrq.lib()
    K = 256
    # R % 4 != 0: the reference's grid R/4 silently drops rows (ops.rs:884)
    R = 6
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(T(wrq, (2 * K * R // 128, 1, 1, 1))),
                              C.byref(V(wrq, (K, 1, 1, 1))), C.byref(V(wrq, (R, 1, 1, 1))), 0, 0)
    assert s == wrq.ERR_ALIGNMENT
    # len % 128 != 0
    s = L.wrq_quantize_mat_int8(None, C.byref(T(wrq, (100, 3, 1, 1))), C.byref(T(wrq, (6, 1, 1, 1))), C.byref(T(wrq, (100, 3, 1, 1))))
    assert s == wrq.ERR_ALIGNMENT
    # chunk kernels: T % 4 (ops.rs:1068-1069)
    R = 8
    s = L.wrq_matmul_mat_int8(None, C.byref(V(wrq, (K, R, 1, 1))), C.byref(T(wrq, (2 * K * R // 128, 1, 1, 1))),
                              C.byref(V(wrq, (K, 6, 1, 1))), C.byref(V(wrq, (R, 6, 1, 1))), 0)
    assert s == wrq.ERR_ALIGNMENT
    # sliced matrix views are refused, not mis-executed
    s = L.wrq_matmul_mat_int8(None, C.byref(V(wrq, (K, R, 1, 1), stride=(K, 2 * R, 1, 1))), C.byref(T(wrq, (2 * K * R // 128, 1, 1, 1))),
                              C.byref(V(wrq, (K, 8, 1, 1))), C.byref(V(wrq, (R, 8, 1, 1))), 0)
    assert s == wrq.ERR_UNSUPPORTED and "sliced matrix views" in err(wrq)
    # ... also a slice that starts inside the parent (the reference's scale indexing has no consistent meaning for it)
    s = L.wrq_matmul_mat_int8(None, C.byref(V(wrq, (K, R, 1, 1), stride=(K, R, 2, 1), offset=(0, 0, 1, 0))), C.byref(T(wrq, (2 * K * R // 128, 1, 1, 1))),
                              C.byref(V(wrq, (K, 8, 1, 1))), C.byref(V(wrq, (R, 8, 1, 1))), 0)
    assert s == wrq.ERR_UNSUPPORTED and "offset 1 along axis 2" in err(wrq)
    # view outside its parent
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(T(wrq, (2 * K * R // 128, 1, 1, 1))),
                              C.byref(V(wrq, (K, 1, 1, 1), stride=(K, 1, 5, 1), offset=(0, 0, 5, 0))), C.byref(V(wrq, (R, 1, 1, 1))), 0, 0)
    assert s == wrq.ERR_SHAPE and "out of range" in err(wrq)
    # dtype outside {F16, F32}, null pointers, unknown activation
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(T(wrq, (2 * K * R // 128, 1, 1, 1))),
                              C.byref(V(wrq, (K, 1, 1, 1), dtype=5)), C.byref(V(wrq, (R, 1, 1, 1))), 0, 0)
    assert s == wrq.ERR_TYPE and err(wrq) == "data type mismatch"
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1), ptr=0)), C.byref(T(wrq, (4, 1, 1, 1))),
                              C.byref(V(wrq, (K, 1, 1, 1))), C.byref(V(wrq, (R, 1, 1, 1))), 0, 0)
    assert s == wrq.ERR_NULL
    s = L.wrq_matmul_vec_int8(None, None, None, None, None, 0, 0)
    assert s == wrq.ERR_NULL
    s = L.wrq_matmul_vec_int8(None, C.byref(T(wrq, (K, R, 1, 1))), C.byref(T(wrq, (2 * K * R // 128, 1, 1, 1))),
                              C.byref(V(wrq, (K, 1, 1, 1))), C.byref(V(wrq, (R, 1, 1, 1))), 99, 0)
    assert s == wrq.ERR_UNSUPPORTED


def test_missing_library_fails_loudly(wrq, monkeypatch, tmp_path):
    monkeypatch.setattr(wrq, "_lib", None)
    monkeypatch.setattr(wrq, "LIB_PATH", str(tmp_path / "nope.so"))
    with pytest.raises(FileNotFoundError, match="no CPU or eager fallback"):
        wrq.lib()


def test_sf4_table_matches_student_quantiles():
    # Float4Quant::new_student (src/tensor/matrix.rs:29-44).  The reference takes the quantile from
    # the statrs crate, which is not available here: the table is checked against scipy's
    # Student-t quantile instead (equal far inside f32) -- bit parity with statrs is unpinned.
    import importlib

    import numpy as np
    from scipy import stats

    wrq = importlib.import_module("web-rwkv_amd")
    delta = (1 / 32 + 1 / 30) / 2
    probs = [delta + (0.5 - delta) / 7 * i for i in range(7)] + [0.5 + (0.5 - delta) / 8 * i for i in range(9)]
    for nu in (1.0, 2.5, 5.0, 30.0):
        q = np.array(wrq.quantile_student(nu), dtype=np.float32)
        ref = stats.t.ppf(probs, nu)
        ref = (ref / ref.max()).astype(np.float32)
        assert q.shape == (16,) and q[0] == -1.0 and q[7] == 0.0 and q[15] == 1.0
        assert (np.diff(q) > 0).all()
        assert np.abs(q.astype(np.float64) - ref.astype(np.float64)).max() <= 1.2e-7


def test_fused_pre_refuses_outputs_over_its_inputs(wrq):
    # a token's workgroup reads its neighbour's row of x and add again while the neighbour stores
    L = wrq.lib()
    Cn, A, row = 64, 3, 64 * 2
    state = C.byref(V(wrq, (Cn, 1, 2, 1), dtype=1))
    far = lambda i: FAKE + 0x1000 * i
    for x, add, ln_out, outs in [(far(1), None, far(1), [far(3)]), (far(1), None, far(2), [far(1) + row]), (far(1), far(2), far(4), [far(2) - 2 * row]),
                                 (far(1), far(2), far(2), [far(5)]), (far(1), None, far(2), [far(3), far(1) + 2 * row])]:
        factors = (C.c_void_p * 2)(far(8), far(8))
        s = L.wrq_fused_pre(None, Cn, A, far(9), x, add, far(6) if add else None, far(7), far(7), 1e-5, state, len(outs), factors, ln_out, (C.c_void_p * 2)(*outs))
        assert s == wrq.ERR_UNSUPPORTED and "overlap no input" in err(wrq), (x, add, ln_out, outs)
        s = L.wrq_v6_pre(None, Cn, A, far(9), x, add, far(6) if add else None, far(7), far(7), 1e-5, state, len(outs), far(8), far(8), ln_out, *(outs + [None])[:2])
        assert s == wrq.ERR_UNSUPPORTED and "overlap no input" in err(wrq)
    s = L.wrq_fused_pre(None, Cn, A, far(9), far(1), far(2), far(1) + row, far(7), far(7), 1e-5, state, 1, (C.c_void_p * 1)(far(8)), far(3), (C.c_void_p * 1)(far(4)))
    assert s == wrq.ERR_UNSUPPORTED and "the sum" in err(wrq)


def test_minor_counts_the_fused_v7_forms(wrq):
    # a binding that calls them asks for this minor: a library of minor 3 may have none of them
    names = [n for n in declared_functions() if n.startswith("wrq_v7_") or n in ("wrq_fused_pre", "wrq_adapters_in")]
    assert len(names) == 7 and wrq.lib().wrq_abi_minor() >= 4
