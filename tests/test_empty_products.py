"""Products over no elements (K = 0): the grouped entry points give ACT(0), whatever the run length and the other products of the call.

The shaders' loops over K are then empty (src/shaders/matmul_vec_int8.wgsl, matmul_vec_nf4.wgsl).  K = 0 satisfies every alignment rule, so
such calls reach the choice of a kernel, which must not hand them to one that divides by its K steps.
"""
import ctypes as C
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def grouped(wrq, kind, Ks, R, T, data, outs, act=0):
    """One grouped call, a product of R rows for every K of `Ks`: f16 activations, f32 outputs, every input at `data`."""
    tensor = lambda *shape: C.pointer(wrq.CTensor(data, shape + (1,) * (4 - len(shape))))
    view = lambda ptr, dtype, *shape: C.pointer(wrq.CTensorView(ptr, wrq.CView(shape + (1, 1), shape + (1, 1), (0, 0, 0, 0)), dtype))
    ops = []
    for K, out in zip(Ks, outs):
        x, o = view(data, wrq.F16, K, T), view(out, wrq.F32, R, T)
        if kind == "int8":
            ops.append(wrq.CVecInt8Op(tensor(K, R), tensor(2 * (K * R // 128)), x, o, act, 0))
        else:
            ops.append(wrq.CVecNf4Op(tensor(K // 2, R), tensor(16), tensor(K * R // 64), x, o, act, 0))
    arr = (type(ops[0]) * len(ops))(*ops)  # keeps the structures it points to alive
    return getattr(wrq.lib(), f"wrq_matmul_vec_{kind}_group")(None, arr, len(ops))


CALLS = [(kind, R, T) for kind in ("int8", "nf4") for R in (64, 4096) for T in (1, 2, 3, 4, 5)]


def test_empty_groups_come_back_without_a_device():
    # in a process of its own that sees no device: nothing can be launched, and a wrong route ends in an integer division by zero
    code = f"""
import importlib, sys
sys.path.insert(0, "tests")
from test_empty_products import CALLS, grouped
wrq = importlib.import_module("web-rwkv_amd")
for kind, R, T in CALLS:
    print(kind, R, T, flush=True)
    status = grouped(wrq, kind, [0], R, T, 0x10000, [0x10000])
    assert status == wrq.ERR_DEVICE, (kind, R, T, status)
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=dict(os.environ, HIP_VISIBLE_DEVICES="-1"), capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, f"exit status {r.returncode} at {r.stdout.splitlines()[-1:]}: {r.stderr[-500:]}"


@pytest.mark.gpu
@pytest.mark.parametrize("kind,R,T", CALLS)
def test_gpu_empty_products(gpu, kind, R, T):
    import torch

    print("empty products on the GPU", kind, R, T, flush=True)
    data = torch.zeros(R * 128, dtype=torch.uint8, device="cuda")
    for Ks in ([0], [128, 0], [0, 128], [0, 0, 128]):
        outs = [torch.full((T, R), float("nan"), device="cuda") for _ in Ks]
        assert grouped(gpu, kind, Ks, R, T, data.data_ptr(), [o.data_ptr() for o in outs], gpu.ACT_SIGMOID) == 0, gpu.lib().wrq_last_error()
        for o in outs:
            assert torch.equal(o, torch.full_like(o, 0.5)), (kind, R, T, Ks)
