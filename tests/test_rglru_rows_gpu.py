"""The recurrent unit's gates and recurrence over many rows (`ops.rglru_rows`) against float64 and beside the kernels one by one, at the
edges of segments and for every size of part."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("blocks,bw,lengths", [(3, 32, [65]), (2, 64, [64, 1, 130]), (1, 128, [128, 0, 70]), (2, 256, [200, 63]),
                                               (9, 32, [700])])
def test_many_rows(dtype, blocks, bw, lengths):
    ops = _ops()
    T, width, B = sum(lengths), blocks * bw, len(lengths)
    u, wide = _rand((T, width), torch.float32, 11), _rand((T, 2 * width), torch.float32, 12)
    weights = (bw ** -0.5 * _rand((2, blocks, bw, bw), torch.float32, 13)).bfloat16().float()
    biases, y_bias = _rand((2, blocks, bw), torch.float32, 14), _rand((width,), torch.float32, 15)
    rate = 0.3 * _rand((width,), torch.float32, 16).abs()
    cu = torch.tensor([sum(lengths[:i]) for i in range(B + 1)], dtype=torch.int32, device=DEV)
    slots = torch.arange(B, 0, -1, dtype=torch.int32, device=DEV)
    held = _rand((B + 1, width + 3), torch.float32, 17)[:, 3:]
    narrow = ops.narrow_gates(weights)
    assert ops.rglru_rows_take(u, narrow, 65) and not ops.rglru_rows_take(u, narrow, 64) and not ops.rglru_rows_take(u, None, 65)
    # in 64 bits
    x = u.double().view(T, blocks, bw)
    r, i = (torch.sigmoid(torch.matmul(x.transpose(0, 1), weights[g].double()).transpose(0, 1) + biases[g].double()).reshape(T, width)
            for g in range(2))
    log_a = -rate.double() * r
    push = torch.sqrt(-torch.expm1(2.0 * log_a)) * i * u.double()
    S_end, states = held.double().clone(), []
    for b in range(B):
        S = S_end[int(slots[b])]
        for t in range(int(cu[b]), int(cu[b + 1])):
            S = torch.exp(log_a[t]) * S + push[t]
            states.append(S)
        S_end[int(slots[b])] = S
    want = torch.stack(states) * torch.nn.functional.gelu(wide[:, :width].double() + y_bias.double(), approximate="tanh")
    off = {}
    for name in ("rows", "kernels"):
        state = held.clone()
        if name == "rows":
            got = ops.rglru_rows(u, narrow, biases, rate, wide[:, :width], y_bias, state, slots, cu, dtype, max(lengths))
        else:
            got = ops.rglru_scan(u, ops.block_gates(u, weights, biases), rate, wide[:, :width], y_bias, state, slots, cu, dtype,
                                 max_q_len=max(lengths))
        assert torch.equal(state[0], held[0])
        off[name] = (float((got.double() - want).norm() / want.norm()), float((state.double() - S_end).norm() / S_end.norm()))
    assert off["rows"][0] <= 1.05 * off["kernels"][0] + 2e-8 and off["rows"][1] <= 1.05 * off["kernels"][1] + 2e-8, off


def test_weights_that_are_left():
    ops = _ops()
    weights = _rand((2, 2, 64, 64), torch.float32, 18).bfloat16().float()
    assert ops.narrow_gates(weights) is not None
    for change in (0.1, float("inf"), float("nan")):
        other = weights.clone()
        other[1, 1, 63, 63] = change
        assert ops.narrow_gates(other) is None
    assert ops.narrow_gates(weights[:, :, :48, :48].contiguous()) is None and ops.narrow_gates(weights.cpu()) is None


def test_an_infinite_input():
    """It reaches the gates of its own part and its own channel's state from its row on, and nothing else."""
    ops = _ops()
    T, blocks, bw = 140, 2, 64
    width = blocks * bw
    u, y = _rand((T, width), torch.float32, 19), _rand((T, width), torch.float32, 20)
    weights = (0.1 * _rand((2, blocks, bw, bw), torch.float32, 21)).bfloat16().float()
    biases, y_bias, rate = (_rand((n,), torch.float32, 22).abs() for n in (2 * width, width, width))
    cu, slots = torch.tensor([0, T], dtype=torch.int32, device=DEV), torch.zeros(1, dtype=torch.int32, device=DEV)
    results = []
    for change in (None, float("inf")):
        if change is not None:
            u[70, 3] = change
        state = torch.zeros((1, width), device=DEV)
        results.append(ops.rglru_rows(u, ops.narrow_gates(weights), biases.view(2, blocks, bw), rate, y, y_bias, state, slots, cu,
                                      torch.float32, T))
    clean, got = results
    assert torch.equal(clean[:70], got[:70]) and torch.equal(clean[:, bw:], got[:, bw:])
    assert not bool(torch.isfinite(got[70, 3]))
