"""Which steps store their values page by page, and float32 steps of many short sequences beside a long one, which do not: the same
numbers in the cache as by the kernel of a wavefront per head."""

import pytest
import torch

from qwen3_from_scratch_amd.ops.build import library


def _dtypes():
    from qwen3_from_scratch_amd import ops

    return ops._DT[torch.bfloat16], ops._DT[torch.float32]


@pytest.mark.parametrize("lengths,D,page,pages", [
    ([512], 128, 16, True), ([512] + [1] * 8, 128, 16, True), ([512] + [1] * 40, 128, 16, False), ([100] + [1] * 60, 128, 16, False),
    ([2048] + [1] * 23, 64, 16, False), ([20] * 30, 64, 16, True), ([8] * 40, 32, 16, True), ([222, 111, 1, 1, 1], 128, 16, True),
    ([7] * 3, 128, 16, False), ([512] + [1] * 40, 128, 64, True)])
def test_float32_steps_that_are_faster_so(lengths, D, page, pages):
    bf16, f32 = _dtypes()
    by_page = library("rotary").q3_values_by_page
    assert bool(by_page(sum(lengths), len(lengths), max(lengths), 8, D, page, f32)) == pages
    assert bool(by_page(sum(lengths), len(lengths), max(lengths), 8, D, page, bf16)) == (max(lengths) >= 8)


@pytest.mark.gpu
@pytest.mark.parametrize("D,page,new", [(32, 16, [90] + [1] * 40), (128, 8, [30, 1, 1, 20] + [1] * 30), (256, 8, [1] * 60 + [40])])
def test_many_short_sequences_beside_a_long_one(D, page, new):
    from test_kernels_gpu import _ops, _rand

    ops = _ops()
    Hq, Hkv, B, T = 4, 2, len(new), sum(new)
    assert not library("rotary").q3_values_by_page(T, B, max(new), Hkv, D, page, _dtypes()[1])
    held = [3 * b for b in range(B)]
    kv = [h + n for h, n in zip(held, new)]
    width = max(-(-n // page) for n in kv)
    pages = torch.randperm(B * width + 1, generator=torch.Generator().manual_seed(1))[:B * width].int().reshape(B, width).cuda()
    cu = torch.tensor([0] + new).cumsum(0).int().cuda()
    seq = torch.repeat_interleave(torch.arange(B), torch.tensor(new)).int().cuda()
    positions = torch.cat([torch.arange(h, h + n) for h, n in zip(held, new)]).int().cuda()
    table = ops.rope_table(1.0 / 10000.0 ** (torch.arange(0, D, 2, device="cuda").float() / D), 512)
    weight, qkv, results = 1.0 + 0.1 * _rand((D,), torch.float32, 2), _rand((T, (Hq + 2 * Hkv) * D), torch.float32, 3), []
    for more in (dict(cu_seqlens_q=cu, kv_lens=torch.tensor(kv).int().cuda(), max_q_len=max(new)), {}):
        rows = qkv.clone()
        keys, values = _rand((B * width + 1, Hkv, page, D), torch.float32, 4), _rand((B * width + 1, Hkv, D, page), torch.float32, 5)
        ops.qk_norm_rope_store(rows, Hq, Hkv, D, positions, seq, q_weight=weight, k_weight=weight, eps=1e-6, table=table, block_table=pages,
                               k_cache=keys, v_cache=values, max_kv_len=max(kv), **more)
        results.append((rows[:, :Hq * D], keys, values))
    for got, want in zip(*results):
        assert torch.allclose(got, want, rtol=2.0 ** -20, atol=2.0 ** -20)      # (a sum of D squares in another order)
    assert torch.equal(results[0][2], results[1][2])
