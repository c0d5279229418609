"""Operands of the fused layer ops that the library cannot check behind a bare pointer (no GPU needed)."""
import pytest
import torch


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
