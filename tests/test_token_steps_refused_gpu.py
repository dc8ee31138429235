"""A Mamba-2 step of single tokens whose norm's weight does not begin at sixteen bytes: the part goes by the kernels one by one, and the
kernels in one refuse before they have moved anything."""

from types import SimpleNamespace

import pytest
import torch

from test_kernels_gpu import _ops, _rand
from test_token_steps_gpu import _step

pytestmark = pytest.mark.gpu


def _off_sixteen(t):
    held = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:]
    held.copy_(t)
    return held


def test_a_part_with_such_a_weight():
    from qwen3_from_scratch_amd.parts.base import Precision
    from qwen3_from_scratch_amd.parts.mamba2 import Mamba2
    from qwen3_from_scratch_amd.weights.random_init import RandomWeights

    part = Mamba2("m", Precision(torch.bfloat16), torch.device("cuda:0"), 64, heads=4, vdim=32, state=32, groups=1, conv=4, norm_groups=1, eps=1e-5)
    source = RandomWeights(part.tensors(), seed=1, std=0.1)
    part.load(lambda name, dtype=None, keep=True: source.get(name, "cuda:0").to(dtype))
    slots, cu, seq = _step(3, 60)
    batch = SimpleNamespace(state_slots=slots, cu_seqlens_q=cu, seq_index=seq, max_q_len=1)
    x, state = _rand((3, 64), torch.bfloat16, 61), _rand((4, part.cache_need().state_shape[0]), torch.float32, 62)
    results = []
    for weight in (part.norm, _off_sixteen(part.norm)):
        part.norm = weight
        held = state.clone()
        results.append((part.forward(x, batch, SimpleNamespace(state=held)), held))
    assert weight.data_ptr() % 16 != 0
    (want, after), (got, held) = results
    assert torch.equal(held, after) and torch.allclose(got.float(), want.float(), rtol=2.0 ** -7, atol=1e-3)


def test_refused_before_anything_moves():
    ops = _ops()
    B, H, P, N, G = 2, 2, 16, 16, 1
    inner, C = H * P, H * P + 2 * G * N
    proj = _rand((B, inner + C + H + 2), torch.bfloat16, 63)[:, :inner + C + H]
    conv, bias = _rand((C, 4), torch.float32, 64), _rand((C,), torch.float32, 65)
    dt_bias, a_log, skip = (_rand((H,), torch.float32, 66 + i) for i in range(3))
    norm, (slots, cu, seq) = _rand((inner,), torch.float32, 69), _step(B, 70)
    state = _rand((B + 1, 3 * C + H * N * P), torch.float32, 71)
    for rows, weight in ((proj, _off_sixteen(norm)), (_rand((B, inner + C + H + 3), torch.bfloat16, 72)[:, 1:1 + inner + C + H], norm)):
        held = state.clone()
        with pytest.raises(ValueError):
            ops.mamba2_token(rows, conv, bias, dt_bias, a_log, skip, weight, 1, 1e-5, held, slots, cu, seq, H, P, N, G)
        assert torch.equal(held, state)
