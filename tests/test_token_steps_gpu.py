"""The recurrent mixers' steps of one token a sequence in fewer kernels, against the kernels one by one: the same numbers, at the edges of
their tiles."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _step(B, seed):
    slots = torch.randperm(B + 1, generator=torch.Generator().manual_seed(seed))[:B].int().to(DEV)
    cu = torch.arange(B + 1, dtype=torch.int32, device=DEV)
    return slots, cu, torch.arange(B, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,P,N,G,parts", [(1, 2, 16, 16, 1, 1), (8, 4, 64, 128, 2, 1), (3, 6, 80, 33, 3, 4), (5, 4, 62, 256, 1, 2),
                                             (2, 64, 64, 65, 1, 1)])
def test_mamba2(dtype, B, H, P, N, G, parts):
    ops = _ops()
    inner, C = H * P, H * P + 2 * G * N
    pad = -(inner + C + H) % 4
    proj = _rand((B, inner + C + H + pad), dtype, 31)[:, :inner + C + H]
    conv, bias = _rand((C, 4), torch.float32, 32), _rand((C,), torch.float32, 33)
    dt_bias, a_log, skip = (_rand((H,), torch.float32, 34 + i) for i in range(3))
    norm = _rand((inner,), torch.float32, 37)
    slots, cu, seq = _step(B, 38)
    held = _rand((B + 1, 3 * C + H * N * P), torch.float32, 39)
    one, two = held.clone(), held.clone()
    xbc = ops.causal_conv(proj[:, inner:inner + C], conv, bias, one[:, :3 * C], slots, cu, seq, activation="silu", out_dtype=dtype,
                          max_q_len=1)
    y = ops.mamba2_scan(xbc, proj[:, inner + C:], dt_bias, a_log, skip, one[:, 3 * C:], slots, cu, H, P, N, G, max_q_len=1)
    want = ops.gated_rmsnorm(y, proj[:, :inner], norm, parts, 1e-5, dtype)
    assert ops.mamba2_token_takes(proj, H, P, N, G, parts, conv, B, B, 1) == ((inner // parts) % 4 == 0)
    if (inner // parts) % 4 == 0:
        got = ops.mamba2_token(proj, conv, bias, dt_bias, a_log, skip, norm, parts, 1e-5, two, slots, cu, seq, H, P, N, G)
        assert torch.equal(got, want) and torch.equal(one, two)


def test_what_mamba2_leaves():
    ops = _ops()
    proj, conv = _rand((3, 32 + 64 + 4), torch.bfloat16, 50), _rand((64, 4), torch.float32, 51)
    takes = [ops.mamba2_token_takes(proj, 4, 8, 16, 1, 1, *args) for args in (
        (conv, 3, 3, 1), (conv, 3, 2, 1), (conv, 3, 3, 2), (conv[:, :3].contiguous(), 3, 3, 1))]
    assert takes == [True, False, False, False]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,blocks,bw", [(1, 1, 4), (8, 8, 256), (17, 3, 30), (20, 2, 321), (16, 4, 16)])
def test_rglru(dtype, B, blocks, bw):
    ops = _ops()
    width = blocks * bw
    u, wide = _rand((B, width), torch.float32, 41), _rand((B, 2 * width), torch.float32, 42)
    weights, biases = 0.1 * _rand((2, blocks, bw, bw), torch.float32, 43), _rand((2, blocks, bw), torch.float32, 44)
    rate, y_bias = _rand((width,), torch.float32, 45).abs(), _rand((width,), torch.float32, 46)
    slots, cu, seq = _step(B, 47)
    held = _rand((B + 1, width + 5), torch.float32, 48)
    one, two = held.clone(), held.clone()
    gates = ops.block_gates(u, weights, biases)
    want = ops.rglru_scan(u, gates, rate, wide[:, :width], y_bias, one[:, 5:], slots, cu, dtype)
    assert ops.rglru_token_takes(u, B, B, 1, blocks) and not ops.rglru_token_takes(u, B, B - 1, 1, blocks)
    got = ops.rglru_token(u, weights, biases, rate, wide[:, :width], y_bias, two[:, 5:], slots, cu, seq, dtype)
    # one kernel's expressions or the other's: a multiply-add that the compiler forms in one and not in the other
    assert torch.allclose(got.float(), want.float(), rtol=2.0 ** -7 if dtype == torch.bfloat16 else 2.0 ** -21, atol=1e-6)
    assert torch.allclose(one, two, rtol=2.0 ** -21, atol=1e-6)
