"""Decoding attention where tiles have no page: what stands in for them is read and never counted."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

BF16 = torch.bfloat16


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("D", [64, 128])
def test_caches_without_a_page(D):
    """Every key and value of a cache without pages counts as zeros, and a step's own are stored nowhere."""
    ops = _ops()
    Hq, Hkv, page = 8, 2, 16
    for lens in ([1, 40], [900, 17]):
        B = len(lens)
        kc, vc = torch.empty((0, Hkv, page, D), dtype=BF16, device="cuda"), torch.empty((0, Hkv, D, page), dtype=BF16, device="cuda")
        bt, cu, kvl = torch.full((B, 64), -1, dtype=torch.int32, device="cuda"), _int32(range(B + 1)), _int32(lens)
        q = _rand((B, Hq, D), BF16, 1)
        for window in (0, 19):
            out = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, 1, max(lens), D ** -0.5, window=window)
            assert torch.equal(out, torch.zeros_like(out))
            out = ops.decode_attention(_rand((B, (Hq + 2 * Hkv) * D), BF16, 2), Hq, Hkv, D, kc, vc, bt, cu, kvl, max(lens),
                                       D ** -0.5, window=window)
            assert torch.equal(out, torch.zeros_like(out))



# every build of the decoding kernel; head sizes and values' sizes of each, with (first) and without a window
BUILDS = [("plain", 64, 64, 0), ("plain", 128, 128, 0), ("plain", 128, 128, 100), ("capped", 128, 128, 0), ("capped", 64, 64, 100),
          ("sigmoid", 64, 64, 0), ("sigmoid", 128, 128, 0), ("pooled", 64, 64, 96), ("pooled", 128, 128, 96),
          ("span", 192, 128, 100), ("span", 96, 64, 0), ("span", 64, 128, 100)]


@pytest.mark.parametrize("build,D,DV,window", BUILDS)
@pytest.mark.parametrize("page", [16, 32])
def test_missing_pages_count_as_zeros(build, D, DV, window, page):
    """Pages given back in the middle, one half of a tile and whole tiles, with NaN in the cache's first page, which
    stands in for them: the bits of the same call over pages of zeros."""
    ops = _ops()
    Hq, Hkv, q_lens, lens, pool = 8, 2, [1, 2, 1, 1, 1], [40, 100, 333, 1500, 2], 4
    B, T = len(lens), sum(q_lens)
    generator = torch.Generator().manual_seed(D + DV + page)

    def paged(longest, seed):
        """Keys and values with NaN in page 0 and zeros in page 1, a table that misses some pages, and the same filled up."""
        counts = [-(-n // page) for n in longest]
        k, v = _rand((sum(counts) + 2, Hkv, page, D), BF16, seed), _rand((sum(counts) + 2, Hkv, DV, page), BF16, seed + 1)
        k[0], v[0], k[1], v[1] = float("nan"), float("nan"), 0.0, 0.0
        table, at = torch.full((B, max(counts) + 2), -1, dtype=torch.int32), 2
        for b, n in enumerate(counts):
            table[b, :n] = torch.arange(at, at + n)
            at += n
        given_back = (torch.rand(table.shape, generator=generator) < 0.4) & (table >= 0)
        return k, v, table.masked_fill(given_back, -1).cuda(), table.masked_fill(given_back, 1).cuda()

    k, v, missing, zeros = paged(lens, 11)
    q = _rand((T, Hq, D), BF16, 13)
    cu, kvl = _int32([0] + torch.tensor(q_lens).cumsum(0).tolist()), _int32(lens)
    more = {"plain": {}, "capped": dict(softcap=30.0), "sigmoid": dict(sigmoid_bias=_rand((Hq,), torch.float32, 14)), "pooled": {},
            "span": dict(span=(0, 40) if window else (256, 20))}[build]
    if build == "pooled":
        rk, rv, runs_missing, runs_zeros = paged([max(1, n // pool) for n in lens], 15)

    def answer(table, runs_table):
        runs = dict(runs=(rk, rv, runs_table, pool)) if build == "pooled" else {}
        return ops.paged_attention(q, Hq, k, v, table, cu, kvl, max(q_lens), max(lens), D ** -0.5, window=window, **more, **runs)

    got = answer(missing, runs_missing if build == "pooled" else None)
    want = answer(zeros, runs_zeros if build == "pooled" else None)
    assert bool(want.isfinite().all()) and bool(want.any())
    assert torch.equal(got, want)
    if build == "plain":
        qkv = _rand((B, (Hq + 2 * Hkv) * D), BF16, 17)
        got, want = (ops.decode_attention(qkv, Hq, Hkv, D, k, v, table, _int32(range(B + 1)), kvl, max(lens), D ** -0.5,
                                          window=window, store=False) for table in (missing, zeros))
        assert bool(want.isfinite().all()) and torch.equal(got, want)
