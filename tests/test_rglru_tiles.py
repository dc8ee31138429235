"""The recurrent unit's rows in tiles of whatever sequence: which steps take them, and many sequences, of no, one and many rows, and segments
whose states a kernel of its own hands on, against float64."""

import pytest
import torch

from qwen3_from_scratch_amd.ops.build import library


@pytest.mark.parametrize("lengths,width,blocks,pays", [
    ([65], 2048, 8, True), ([65] + [1] * 23, 2048, 8, True), ([65] + [1] * 40, 2048, 8, False), ([128] + [1] * 64, 2048, 8, False),
    ([512] + [1] * 40, 2048, 8, True), ([512] + [1] * 64, 2048, 8, False), ([1024] + [1] * 64, 2048, 8, True), ([2048] + [1] * 40, 2048, 8, True),
    ([66] + [10] * 63, 2048, 8, False), ([65] * 64, 2048, 8, True), ([512] + [1] * 23, 4096, 16, True), ([512] + [1] * 40, 4096, 16, False),
    ([512] + [1] * 40, 2048, 32, True), ([2048] + [1] * 40, 1024, 32, True), ([32768], 2048, 8, True), ([512], 2048, 2, False)])
def test_steps_that_are_faster_so(lengths, width, blocks, pays):
    assert bool(library("rglru").q3_rglru_rows_pay(sum(lengths), len(lengths), width, blocks)) == pays


@pytest.mark.gpu
@pytest.mark.parametrize("blocks,bw,lengths", [
    (2, 32, [66] + [1] * 62 + [70, 0, 130]),             # the sixty-fourth sequence and those behind it
    (1, 64, [0, 0, 65, 1, 64, 128, 0]), (2, 32, [1] * 130 + [200]),
    (1, 32, [4097, 31, 0, 4500]), (1, 64, [5000])])      # states handed on by a kernel of its own
def test_tiles_of_many_sequences(blocks, bw, lengths):
    from test_kernels_gpu import _ops, _rand

    ops = _ops()
    T, width, B = sum(lengths), blocks * bw, len(lengths)
    u, wide = _rand((T, width), torch.float32, 81), _rand((T, 2 * width), torch.float32, 82)
    weights = (bw ** -0.5 * _rand((2, blocks, bw, bw), torch.float32, 83)).bfloat16().float()
    biases, y_bias = _rand((2, blocks, bw), torch.float32, 84), _rand((width,), torch.float32, 85)
    rate = 0.3 * _rand((width,), torch.float32, 86).abs()
    ends = torch.tensor([0] + lengths).cumsum(0).tolist()
    cu = torch.tensor(ends, dtype=torch.int32, device="cuda")
    slots = torch.randperm(B + 1, generator=torch.Generator().manual_seed(87))[:B].int().cuda()
    held = _rand((B + 1, width), torch.float32, 88)
    x = u.double().view(T, blocks, bw)
    r, i = (torch.sigmoid(torch.matmul(x.transpose(0, 1), weights[g].double()).transpose(0, 1) + biases[g].double()).reshape(T, width)
            for g in range(2))
    log_a = -rate.double() * r
    decay, push = torch.exp(log_a).cpu(), (torch.sqrt(-torch.expm1(2.0 * log_a)) * i * u.double()).cpu()
    S_end, states = held.double().cpu(), torch.empty(T, width, dtype=torch.float64)
    for b in range(B):
        S = S_end[int(slots[b])]
        for t in range(ends[b], ends[b + 1]):
            S = decay[t] * S + push[t]
            states[t] = S
        S_end[int(slots[b])] = S
    branch = torch.nn.functional.gelu(wide[:, :width].double() + y_bias.double(), approximate="tanh").cpu()
    state = held.clone()
    got = ops.rglru_rows(u, ops.narrow_gates(weights), biases, rate, wide[:, :width], y_bias, state, slots, cu, torch.float32, max(lengths))
    # float32 throughout: some ten roundings of 2^-24 in a gate, and as many again where a state is carried on
    for found, want in ((got, states * branch), (state, S_end)):
        assert float((found.double().cpu() - want).norm() / want.norm()) <= 32 * 2.0 ** -24
        assert bool(((found.double().cpu() - want).abs() <= 1e-4 * (want.abs() + 1.0)).all())
