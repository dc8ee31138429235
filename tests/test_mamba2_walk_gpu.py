"""Mamba-2's recurrence over many bfloat16 rows (`ops.mamba2_scan`) against float64, at the edges of its chunks, its tiles of columns
and its sizes of state."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _inputs(H, P, N, G, lengths, seed):
    T, C = sum(lengths), H * P + 2 * G * N
    xbc, wide = _rand((T, C), torch.bfloat16, seed), _rand((T, H + 3), torch.bfloat16, seed + 1)
    cu = torch.tensor([sum(lengths[:i]) for i in range(len(lengths) + 1)], dtype=torch.int32, device=DEV)
    slots = torch.tensor(list(range(len(lengths), 0, -1)), dtype=torch.int32, device=DEV)
    state = _rand((len(lengths) + 1, 5 + H * N * P), torch.float32, seed + 2)[:, 5:]
    dt_bias, a_log, skip = (_rand((H,), torch.float32, seed + 3 + i) for i in range(3))
    return xbc, wide[:, 3:], dt_bias, a_log, skip, state, slots, cu


def _exact(xbc, dt, dt_bias, a_log, skip, state, slots, cu, H, P, N, G):
    state, y = state.double().clone(), []
    for b, slot in enumerate(slots.tolist()):
        S = state[slot].reshape(H, N, P)
        for t in range(int(cu[b]), int(cu[b + 1])):
            x, B, C = xbc[t].double().split((H * P, G * N, G * N))
            x = x.view(H, P)
            B, C = (m.view(G, N).repeat_interleave(H // G, dim=0) for m in (B, C))
            step = torch.nn.functional.softplus(dt[t].double() + dt_bias.double())
            S = torch.exp(-torch.exp(a_log.double()) * step)[:, None, None] * S + (step[:, None] * B)[:, :, None] * x[:, None, :]
            y.append((S * C[:, :, None]).sum(dim=1) + skip.double()[:, None] * x)
        state[slot] = S.reshape(-1)
    return torch.stack(y).reshape(len(y), H * P), state


@pytest.mark.parametrize("H,P,N,G,lengths", [(2, 16, 32, 1, [9]), (4, 64, 128, 2, [64, 1, 65]), (3, 80, 64, 3, [63, 0, 130, 7]),
                                             (70, 32, 32, 1, [128, 11]), (2, 48, 256, 1, [200])])
def test_many_rows(H, P, N, G, lengths):
    ops = _ops()
    xbc, dt, dt_bias, a_log, skip, state, slots, cu = _inputs(H, P, N, G, lengths, 70)
    want, after = _exact(xbc, dt, dt_bias, a_log, skip, state, slots, cu, H, P, N, G)
    off = {}
    for name, rows in (("walk", xbc), ("float32", xbc.float())):      # the float32 rows take the float32 chunks' kernels
        held = state.clone()
        y = ops.mamba2_scan(rows, dt if name == "walk" else dt.float(), dt_bias, a_log, skip, held, slots, cu, H, P, N, G,
                            max_q_len=max(lengths))
        assert y.dtype == torch.float32
        off[name] = (float((y.double() - want).norm() / want.norm()), float((held.double() - after).norm() / after.norm()))
        assert torch.equal(held[0], state[0])                          # a slot of nobody's
    # the same sums with fewer roundings; decays' logarithms of up to 64 rows add up in float32 in both
    assert off["walk"][0] <= 1.1 * off["float32"][0] + 1e-7 and off["walk"][1] <= 1.1 * off["float32"][1] + 1e-7, off
    assert off["walk"][0] <= 1e-6


def test_rows_that_are_no_numbers():
    """An infinite x stays one in its own column and head, and the state that it leaves; other columns and sequences stay as they are, and so
    do the chunks before it. (In its own column the rows before it, in its chunk, may be no numbers: what they multiply it with is zero.)"""
    ops = _ops()
    H, P, N, G, lengths = 2, 32, 64, 1, [70, 12]
    xbc, dt, dt_bias, a_log, skip, state, slots, cu = _inputs(H, P, N, G, lengths, 90)
    clean, held = ops.mamba2_scan(xbc, dt, dt_bias, a_log, skip, state.clone(), slots, cu, H, P, N, G, max_q_len=70), state.clone()
    xbc[66, 3] = float("inf")
    xbc[66, H * P:H * P + N] = xbc[66, H * P:H * P + N].abs() + 0.5
    got = ops.mamba2_scan(xbc, dt, dt_bias, a_log, skip, held, slots, cu, H, P, N, G, max_q_len=70)
    assert torch.equal(got[:64], clean[:64]) and torch.equal(got[70:], clean[70:])
    assert not bool(torch.isfinite(got[66:70, 3]).any()) and bool(torch.isfinite(got[64:70, 32:]).all())
    last = held[2].view(H, N, P)
    assert bool((last[0, :, 3] == float("inf")).all()) and bool(torch.isfinite(last[1]).all())
