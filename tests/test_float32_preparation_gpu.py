"""Queries, keys and values of float32 steps prepared in 16-byte accesses, against the kernel of a wavefront per head (which a step whose
sequences are not described takes): head sizes, pages, sequences that begin and end inside a page, rows off sixteen bytes."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("weights", ["float32", "bfloat16", None])
@pytest.mark.parametrize("D,page,held,new", [(16, 8, [0, 5], [3, 7]), (32, 16, [15, 0, 40], [9, 1, 33]), (64, 64, [60], [70]),
                                             (128, 16, [0, 149, 31], [201, 1, 17]), (256, 32, [3], [8])])
def test_float32_steps(weights, D, page, held, new):
    ops = _ops()
    Hq, Hkv, B, T = 6, 3, len(new), sum(new)
    qkv = _rand((T, (Hq + 2 * Hkv) * D), torch.float32, 21)
    w = [1.0 + 0.2 * _rand((D,), torch.float32, 22 + i) for i in range(2)] if weights else [None, None]
    if weights == "bfloat16":
        w = [x.bfloat16() for x in w]
    table = ops.rope_table(1.0 / 10000.0 ** (torch.arange(0, D, 2, device=DEV).float() / D), 512)
    kv = [h + n for h, n in zip(held, new)]
    width = max(-(-n // page) for n in kv)
    pages = torch.randperm(B * width + 1, generator=torch.Generator().manual_seed(23))[:B * width].int().reshape(B, width).to(DEV)
    pages[B - 1, width - 1] = -1                # a page that is not there: its tokens are stored nowhere
    cu = torch.tensor([sum(new[:i]) for i in range(B + 1)], dtype=torch.int32, device=DEV)
    seq = torch.cat([torch.full((n,), b) for b, n in enumerate(new)]).int().to(DEV)
    positions = torch.cat([torch.arange(h, h + n) for h, n in zip(held, new)]).int().to(DEV)
    lens = torch.tensor(kv, dtype=torch.int32, device=DEV)
    results = []
    for described, off in ((True, 0), (False, 0), (True, 1)):
        rows = torch.empty(T * (Hq + 2 * Hkv) * D + off, device=DEV)[off:].view(T, -1).copy_(qkv)
        keys = _rand((B * width + 1, Hkv, page, D), torch.float32, 24)
        values = _rand((B * width + 1, Hkv, D, page), torch.float32, 25)
        more = dict(cu_seqlens_q=cu, kv_lens=lens, max_q_len=max(new)) if described else {}
        ops.qk_norm_rope_store(rows, Hq, Hkv, D, positions, seq, q_weight=w[0], k_weight=w[1], eps=1e-6, table=table,
                               block_table=pages, k_cache=keys, v_cache=values, max_kv_len=max(kv), **more)
        results.append((rows[:, :Hq * D].clone(), keys, values))
    for fast, general, aside in zip(*results):
        assert torch.equal(general, aside)
        # a sum of D squares in another order, then three products and a sum: a few units in the last place of the pair's size
        assert torch.allclose(fast, general, rtol=2.0 ** -20, atol=2.0 ** -20)
    assert torch.equal(results[0][2], results[1][2])
