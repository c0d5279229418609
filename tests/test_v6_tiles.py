"""The second halves of a v6 layer's adapters in both forms: a token at a time and in tiles of 16 channels x 16 tokens, at the
edges of the tiles and of the rule between them, against float64."""
import importlib
import os
import sys

import numpy as np
import pytest

from helpers import assert_close

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
@pytest.mark.parametrize("C", [16, 80, 100, 256])
@pytest.mark.parametrize("runs", [[(1, 7)], [(0, 3), (2, 5)], [(2, 1)] + [(1, 15)], [(0, 17)], [(2, 20), (0, 1), (1, 16)]], ids=lambda r: str(sum(n for _, n in r)))
@pytest.mark.parametrize("mix_lora,decay_lora", [(32, 64), (64, 128)])
def test_gpu_v6_tiles(gpu, C, runs, mix_lora, decay_lora):
    import torch

    sys.path.insert(0, ROOT)
    lop = importlib.import_module("oracle.layer_ops")
    print("v6 adapter tiles on the GPU", C, runs, mix_lora, decay_lora, flush=True)
    B = 3
    cur = lop.pack_cursors(runs)
    A = len(cur)
    g = torch.Generator().manual_seed(0x5754 + C + A)
    h = lambda *s, std=0.3: (torch.randn(s, generator=g) * std).half()
    lora, w2, mix, x = h(A, 5, mix_lora, std=0.5), h(5, C, mix_lora, std=0.1), torch.rand((5, C), generator=g).half(), h(A, C, std=1.0)
    state = torch.randn((B, 66, C), generator=g)
    dl, dw2, bias = h(A, decay_lora, std=0.5), h(C, decay_lora, std=0.1), h(C, std=0.5)
    curd = torch.from_numpy(cur.view(np.int32)).cuda()
    out, decay = torch.empty((5, A, C), dtype=torch.float16, device="cuda"), torch.empty((A, C), dtype=torch.float32, device="cuda")
    gpu.FusedV6.time_mix(C, A, mix_lora, curd, lora.cuda(), w2.cuda(), mix.cuda(), state.cuda(), ((C, 65, B), (C, 66, B), (0, 0, 0)), x.cuda(), out)
    gpu.FusedV6.decay(C, A, decay_lora, dl.cuda(), dw2.cuda(), bias.cuda(), decay)
    prev = torch.cat([x[:1], x[:-1]]).double()
    at = 0
    for slot, n in runs:
        prev[at] = state[slot, 0].double()
        at += n
    f = torch.einsum("ask,sck->sac", lora.double(), w2.double()) + mix.double()[:, None]
    want = x.double() * (1 - f) + prev * f
    # f passes through two f16 roundings (2^-11 of values up to 4 each) and meets |x| + |prev| up to 8; the output is rounded once more
    assert_close(out.cpu().numpy(), want.numpy(), 1.6e-2, "time_mix vs float64")
    assert float((out.cpu().double() - want).norm() / want.norm()) < 1e-3  # 2^-11 per rounding, three of them
    want = torch.exp(-torch.exp(dl.double() @ dw2.double().t() + bias.double()))
    assert_close(decay.cpu().numpy(), want.numpy(), 2e-6, "decay vs float64")  # sums of 128 terms in f32, two exponentials


@pytest.mark.gpu
@pytest.mark.parametrize("C", [32, 2080, 2592, 4128, 8192])
@pytest.mark.parametrize("A", [1, 17])
def test_gpu_adapters_in_long_rows(gpu, C, A):
    """First halves of adapters either side of the sizes where waves and steps in flight change."""
    import torch

    print("adapters_in on the GPU", C, A, flush=True)
    g = torch.Generator().manual_seed(0x5755 + C + A)
    h = lambda *s: (torch.randn(s, generator=g) * 0.05).half()
    ops = [(h(16, C), h(A, C), torch.empty((A, 16), dtype=torch.float16, device="cuda"), gpu.ACT_NONE),
           (h(48, C), h(A, C), torch.empty((A, 48), dtype=torch.float16, device="cuda"), gpu.ACT_TANH)]
    gpu.FusedV7.adapters_in(C, A, [(w.cuda(), x.cuda(), out, act) for w, x, out, act in ops])
    for w, x, out, act in ops:
        want = x.double() @ w.double().t()
        want = torch.tanh(want) if act == gpu.ACT_TANH else want
        # f32 sums of up to 8192 products of 2.5e-3 each, one rounding to f16 (2^-11) of values below 1
        assert_close(out.cpu().numpy(), want.numpy(), 1e-3, "adapters_in vs float64")


@pytest.mark.gpu
@pytest.mark.parametrize("C", [128, 768, 1152, 2048, 2176, 4224])
@pytest.mark.parametrize("A", [1, 15, 16, 33])
def test_gpu_adapters_in_lines(gpu, C, A):
    """First halves of adapters over channels in whole steps of 128: fewer steps than waves, one round of two steps per wave, more."""
    import torch

    print("adapters_in in lines on the GPU", C, A, flush=True)
    g = torch.Generator().manual_seed(0x575A + C + A)
    h = lambda *s: (torch.randn(s, generator=g) * 0.05).half()
    ops = [(h(r, C), h(A, C), torch.empty((A, r), dtype=torch.float16, device="cuda"), act) for r, act in ((32, gpu.ACT_NONE), (16, gpu.ACT_SIGMOID), (80, gpu.ACT_NONE))]
    gpu.FusedV7.adapters_in(C, A, [(w.cuda(), x.cuda(), out, act) for w, x, out, act in ops])
    for w, x, out, act in ops:
        want = x.double() @ w.double().t()
        want = torch.sigmoid(want) if act == gpu.ACT_SIGMOID else want
        # f32 sums of up to 4224 products of 2.5e-3 each, one rounding to f16 (2^-11) of values below 1
        assert_close(out.cpu().numpy(), want.numpy(), 1e-3, "adapters_in vs float64")


@pytest.mark.gpu
@pytest.mark.parametrize("C", [2112, 2144, 2528, 2592, 4256, 4320, 5088, 5184, 5216])
@pytest.mark.parametrize("A", [1, 33])
def test_gpu_adapters_in_gathered(gpu, C, A):
    """First halves of adapters over channels in no whole steps of 128, either side of the lines between their three forms: one round of
    eight or ten steps per wave, more, sixteen waves."""
    import torch

    print("adapters_in gathered on the GPU", C, A, flush=True)
    g = torch.Generator().manual_seed(0x575B + C + A)
    h = lambda *s: (torch.randn(s, generator=g) * 0.05).half()
    ops = [(h(r, C), h(A, C), torch.empty((A, r), dtype=torch.float16, device="cuda"), act) for r, act in ((48, gpu.ACT_NONE), (16, gpu.ACT_SIGMOID))]
    gpu.FusedV7.adapters_in(C, A, [(w.cuda(), x.cuda(), out, act) for w, x, out, act in ops])
    for w, x, out, act in ops:
        want = x.double() @ w.double().t()
        want = torch.sigmoid(want) if act == gpu.ACT_SIGMOID else want
        # f32 sums of up to 5216 products of 2.5e-3 each, one rounding to f16 (2^-11) of values below 1
        assert_close(out.cpu().numpy(), want.numpy(), 1e-3, "adapters_in vs float64")


@pytest.mark.gpu
def test_gpu_pre_of_one_token_in_place(gpu):
    """A single token has no neighbour that reads its row: normalised in place as into a buffer of its own."""
    import torch

    C = 4100
    g = torch.Generator().manual_seed(0x5759)
    h = lambda *s: torch.randn(s, generator=g).half().cuda()
    cur, state, view = torch.tensor([1 << 24], dtype=torch.int32).cuda(), torch.randn((1, 1, C), generator=g).cuda(), ((C, 1, 1), (C, 1, 1), (0, 0, 0))
    x, w, b, f, ln, out = (h(C) for _ in range(6))
    args = lambda x, ln, out: (C, 1, cur, x, None, None, w, b, 1e-5, state, view, [f], ln, [out])
    gpu.FusedV7.pre(*args(x, ln, out))
    again, shifted = x.clone(), torch.empty_like(out)
    gpu.FusedV7.pre(*args(again, again, shifted))
    assert torch.equal(again, ln) and torch.equal(shifted, out)
