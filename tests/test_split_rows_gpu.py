"""Decoding attention whose keys several blocks shared out, merged inside the product that reads it."""

import pytest
import torch

from test_kernels_gpu import _ops, _paged_case, _rand

pytestmark = pytest.mark.gpu


def _merged(parts):
    """The rows in float64, from the partial results."""
    S, B, Hkv, D, G = parts.splits, parts.rows, parts.kv_heads, parts.dim, parts.heads // parts.kv_heads
    n = B * Hkv * S * 16
    acc = parts.workspace[:n * D].view(B, Hkv, S, 16, D)[:, :, :, :G].double()
    ml = parts.workspace[n * D:].view(B, Hkv, S, 16, 2)[:, :, :, :G].double()
    weight = torch.exp2(ml[..., 0] - ml[..., 0].amax(2, keepdim=True)).unsqueeze(-1)
    return ((weight * acc).sum(2) / (weight * ml[..., 1:]).sum(2)).reshape(B, -1)


# a wavefront's share of K of 256, 512 and 1,024 numbers, idle wavefronts, one head a key head and sixteen, keys for four parts
# and for thirty-two (sixteen are made), sequences so much shorter than the longest that most of their parts are empty; the last
# needs more shared memory than a block gets unasked
@pytest.mark.parametrize("Hq,Hkv,D,N,kv_lens", [
    (16, 8, 128, 1024, [1101]), (16, 8, 128, 1024, [5000]), (32, 8, 128, 4096, [500]), (64, 8, 128, 32, [300]),
    (16, 8, 128, 1040, [500, 3]), (4, 1, 64, 64, [600, 1, 65, 300]), (16, 1, 64, 16, [2500]), (2, 2, 128, 48, [400] * 15),
    (36, 4, 64, 208, [450, 300]), (8, 2, 128, 512, [600] * 3), (36, 18, 64, 96, [600] * 7)])
@pytest.mark.parametrize("norm_dtype,window", [(torch.float32, 0), (torch.bfloat16, 23)])
def test_the_product_merges_what_the_blocks_left(Hq, Hkv, D, N, kv_lens, norm_dtype, window):
    ops = _ops()
    B, K = len(kv_lens), Hq * D
    _, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, B, Hq, Hkv, D, 16, [1] * B, kv_lens, 21)
    qkv = _rand((B, (Hq + 2 * Hkv) * D), torch.bfloat16, 22, scale=1.5)
    weight = _rand((N, K), torch.bfloat16, 23, scale=K ** -0.5)
    residual = _rand((B, N), torch.float32, 24)
    norm = (1.0 + _rand((N,), torch.float32, 25, scale=0.3)).to(norm_dtype)
    args = (Hq, Hkv, D, kc, vc, bt, cu, kvl, max(kv_lens), D ** -0.5)
    parts = ops.decode_attention(qkv, *args, window=window, residual_width=N)
    assert isinstance(parts, ops.SplitRows) and 2 <= parts.splits <= 16
    x = _merged(parts)
    # (the rows are what the kernel gives that merges them itself, to bfloat16's half unit beside float32 sums)
    rows = ops.decode_attention(qkv, *args, window=window)
    torch.testing.assert_close(x, rows.double(), rtol=2.0 ** -7, atol=1e-3)
    new = residual.clone()
    values, sums = ops.linear_residual_norm(parts, weight, ops.tile_weight(weight), new, norm)

    # float32 merging is within 2^-18 of x: where that is enough to round another way, either result is right
    low, high = ((x * (1 + e)).float().bfloat16().double() for e in (-2.0 ** -18, 2.0 ** -18))
    w = weight.double()
    size = x.abs() @ w.abs().t()
    want = low @ w.t()
    slack = (high - low).abs() @ w.abs().t() + K * 2.0 ** -24 * size
    # the product in bfloat16 (half a unit: 2^-8 of it), the sum in float32
    bound = slack + 2.0 ** -8 * (want.abs() + slack) + 2.0 ** -23 * (residual.double().abs() + want.abs() + slack)
    assert ((new.double() - residual.double() - want).abs() <= bound).all()
    torch.testing.assert_close(values.float(), new * norm.float(), rtol=2.0 ** -8, atol=0)
    torch.testing.assert_close(sums.sum(0)[:B], (new ** 2).sum(1), rtol=1e-5, atol=0)


@pytest.mark.parametrize("Hq,kv_lens", [(32, [2060] * 2), (16, [8193])])
def test_partial_results_too_many_to_read_in_every_block_are_merged_first(Hq, kv_lens):
    ops = _ops()
    B, Hkv, D = len(kv_lens), 8, 128
    _, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, B, Hq, Hkv, D, 16, [1] * B, kv_lens, 26)
    qkv = _rand((B, (Hq + 2 * Hkv) * D), torch.bfloat16, 27)
    args = (Hq, Hkv, D, kc, vc, bt, cu, kvl, max(kv_lens), D ** -0.5)
    got = ops.decode_attention(qkv, *args, residual_width=4096)
    assert torch.equal(got, ops.decode_attention(qkv, *args))


def test_an_infinite_value_stays_one():
    """An infinity among the values of the last of ten parts, which are merged in steps of eight: as merged beforehand."""
    ops = _ops()
    B, Hq, Hkv, D, N, keys = 12, 2, 2, 128, 64, 2000
    _, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, B, Hq, Hkv, D, 16, [1] * B, [keys] * B, 28)
    qkv, weight = _rand((B, (Hq + 2 * Hkv) * D), torch.bfloat16, 29), _rand((N, Hq * D), torch.bfloat16, 30, scale=0.05)
    args = (Hq, Hkv, D, kc, vc, bt, cu, kvl, keys, D ** -0.5)
    splits = ops.decode_attention(qkv, *args, residual_width=N).splits
    assert splits == 10
    key = 32 * 4 * (splits - 1)                # a wavefront's tiles of 32 keys: every (4 splits)-th, from this one on
    vc[int(bt[3, key // 16]), 1, 5, key % 16] = float("inf")
    norm, results = torch.ones(N, device="cuda"), []
    for width in (N, 0):
        rows, residual = ops.decode_attention(qkv, *args, residual_width=width), torch.zeros(B, N, device="cuda")
        ops.linear_residual_norm(rows, weight, ops.tile_weight(weight), residual, norm)
        results.append(residual)
    assert bool(results[1][3].isinf().all()) and bool(results[1].isfinite()[torch.arange(B) != 3].all())
    assert torch.equal(results[0][3], results[1][3]) and bool(results[0].isfinite()[torch.arange(B) != 3].all())
