"""Products that carry a norm by the kernel that shares K out inside a block, at the edges of its tiles."""

import pytest
import torch

from test_kernels_gpu import _forget_choices, _ops, _rand, rules_alone

pytestmark = pytest.mark.gpu


# every shape of the dispatch (by its number), at rows and columns that end inside a tile, and inner sizes that leave
# groups without a stage, with a short share and with an uneven one
@pytest.mark.parametrize("M,N,K,shape", [(17, 4096, 64, 0), (17, 1028, 8640, 0), (33, 4084, 192, 1), (64, 4096, 1024, 1), (100, 4092, 1344, 2),
                                         (65, 8188, 1024, 3), (201, 8188, 320, 4), (257, 8180, 1088, 5), (640, 4100, 2176, 5),
                                         (128, 32764, 1088, 5)])
def test_products_that_carry_a_norm(M, N, K, shape):
    ops = _ops()
    assert ops.matmul_fused_plan("scaled", M, N, K) == (16 + shape, 1)
    x, w = _rand((M, K), torch.bfloat16, 91), _rand((N, K), torch.bfloat16, 92, scale=0.05)
    sums = (0.5 + torch.rand((37, ops.sums_stride(M)), generator=torch.Generator().manual_seed(93))).cuda() * K / 37
    eps = 1e-5
    factor = torch.rsqrt(sums[:, :M].double().sum(dim=0) / K + eps)[:, None]
    exact = (x.double() @ w.double().T) * factor
    # K products of bfloat16 numbers summed in float32, K roundings of 2^-24 of the sum of the magnitudes at most, and the
    # factor's few
    bound = (K + 64) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) * factor
    got = ops.linear(x, w, out_dtype=torch.float32, unscaled=(sums, eps, K))
    assert bool(((got.double() - exact).abs() <= bound).all())
    assert torch.equal(ops.linear(x, w, unscaled=(sums, eps, K)), got.bfloat16())
    assert torch.equal(ops.linear_swiglu(x, w, unscaled=(sums, eps, K)), ops.swiglu(got.bfloat16()))


@pytest.mark.parametrize("norm_dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,columns", [(65, 1024, 2048, 16), (129, 1012, 4096, 32), (400, 1024, 1088, 32), (640, 1016, 3200, 64),
                                           (300, 4100, 320, 128)])
def test_residual_addition_and_the_next_norm(M, N, K, columns, norm_dtype):
    ops = _ops()
    x, w = _rand((M, K), torch.bfloat16, 94), _rand((N, K), torch.bfloat16, 95, scale=0.05)
    nw = (1.0 + _rand((N,), torch.float32, 96, scale=0.2)).to(norm_dtype)
    residual = _rand((M, N), torch.float32, 97, scale=2.0)
    exact = x.double() @ w.double().T
    stream = residual.clone()
    values, sums = ops.linear_residual_norm(x, w, None, stream, nw)
    assert sums.shape == (-(-N // columns), ops.sums_stride(M))
    # the product rounded to bfloat16 once, from a float32 sum that is off by what its additions round
    delta = (stream - residual).double()
    bound = 2.0 ** -8 * exact.abs() + (K + 64) * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -23 * stream.double().abs()
    assert bool(((delta - exact).abs() <= bound).all())
    assert torch.equal(values, (stream * nw.float()).bfloat16())
    torch.testing.assert_close(sums[:, :M].double().sum(dim=0), (stream.double() ** 2).sum(dim=1), rtol=1e-5, atol=1e-6)
    again = residual.clone()
    v2, s2 = ops.linear_residual_norm(x, w, None, again, nw)
    assert torch.equal(again, stream) and torch.equal(v2, values) and torch.equal(s2[:, :M], sums[:, :M])


def test_rows_that_two_kernels_take():
    """17 to 64 rows of a small weight: from 4,096 columns on not the few-row kernel, with its bits."""
    ops = _ops()
    for N, M in ((4096, 17), (4096, 64), (8192, 32), (1024, 64)):
        torch.manual_seed(100)
        x, w = _rand((M, 1024), torch.bfloat16, 98), _rand((N, 1024), torch.bfloat16, 99, scale=0.05)
        tiled, sums = ops.tile_weight(w), torch.rand((64, ops.sums_stride(M)), device="cuda") * 32.0
        got = ops.linear(x, w, out_dtype=torch.float32, tiled=tiled, unscaled=(sums, 1e-5, 1024))
        by_tiles = ops.linear(x, w, out_dtype=torch.float32, unscaled=(sums, 1e-5, 1024))
        assert bool(ops._groups_before_few(w, M, (sums, 1e-5, 1024))) == (N >= 4096)
        assert not ops._groups_before_few(w, 16, (sums, 1e-5, 1024)) and not ops._groups_before_few(w, M, None)
        torch.testing.assert_close(got, by_tiles, rtol=1e-4, atol=1e-4)
        first = ops.linear(x[:16].contiguous(), w, out_dtype=torch.float32, tiled=tiled, unscaled=(sums[:, :16].contiguous(), 1e-5, 1024))
        assert torch.equal(first, got[:16])
    w = _rand((4096, 2048), torch.bfloat16, 99)          # eight shares of K there, four here
    assert not ops._groups_before_few(w, 32, (sums, 1e-5, 2048))


@pytest.mark.parametrize("kind,other", [("scaled_swiglu", "scaled"), ("scaled", "scaled_swiglu")])
def test_a_table_entry_for_one_of_the_two_epilogues(rules_alone, kind, other):
    """A size that the table sends to the tiles, with the activation or without: the few-row kernel keeps its rows there, and
    either way a row's bits are those it has among sixteen."""
    ops, (M, N, K) = rules_alone, (32, 4096, 1024)
    ops.matmul_table([{"kind": kind, "rows": M, "N": N, "K": K, "own": 1, "splits": 8}], clear=True)
    _forget_choices(ops)
    x, w = _rand((M, K), torch.bfloat16, 98), _rand((N, K), torch.bfloat16, 99, scale=0.05)
    tiled, sums = ops.tile_weight(w), torch.rand((64, M), generator=torch.Generator().manual_seed(97)).cuda() * 32.0
    products = {"scaled": lambda x, sums: ops.linear(x, w, out_dtype=torch.float32, tiled=tiled, unscaled=(sums, 1e-5, K)),
                "scaled_swiglu": lambda x, sums: ops.linear_swiglu(x, w, tiled=tiled, unscaled=(sums, 1e-5, K))}
    unscaled = (sums, 1e-5, K)
    assert not ops._groups_before_few(w, M, unscaled, kind == "scaled_swiglu")
    assert ops._groups_before_few(w, M, unscaled, other == "scaled_swiglu")
    for product in products.values():
        assert torch.equal(product(x, sums)[:16], product(x[:16].contiguous(), sums[:, :16].contiguous()))


def test_the_tuner_finds_these_kernels_and_a_table_names_them(rules_alone):
    """Where they are the fastest by far the contest ends with them, what it found goes into a table, and a table that says
    otherwise is followed, plain products of one round of tiles among them."""
    from qwen3_from_scratch_amd.ops import tune

    ops = rules_alone
    ops.matmul_candidates(1)
    try:
        small, large = tune.tune_layer(1024, 16, 8, 128, 4096, [201]), tune.tune_layer(4096, 32, 8, 128, 1024, [535])
    finally:
        ops.matmul_candidates(16)
    found = {(e["kind"], e["N"], e["K"]): e for e in small + large}
    carrying = [("scaled", 4096, 1024), ("scaled_swiglu", 8192, 1024), ("residual", 1024, 2048), ("residual", 1024, 4096)]
    rules = [ops.matmul_fused_plan(kind, 201, N, K) for kind, N, K in carrying]
    assert [(found[c].get("own"), found[c].get("splits")) for c in carrying] == rules and all(own >= 16 for own, _ in rules)
    assert found["plain_round", 4096, 4096]["own"] == 32 + 9 and ("plain", 4096, 4096) not in found

    x, w = _rand((535, 4096), torch.bfloat16, 31), _rand((4096, 4096), torch.bfloat16, 32, scale=0.05)
    want = x.double() @ w.double().T
    others = [dict(e, **other) for e, other in ((found["scaled", 4096, 1024], dict(own=18)),
                                               (dict(found["plain_round", 4096, 4096], library=0), dict(own=-1)))]
    for table, scaled, plain in ((list(found.values()), rules[0][0], 32 + 9), (others, 18, -1)):
        ops.matmul_table(table, clear=True)
        _forget_choices(ops)
        assert ops.matmul_fused_plan("scaled", 201, 4096, 1024) == (scaled, 1)
        torch.testing.assert_close(ops.linear(x, w).double(), want, rtol=1.6e-2, atol=5e-2)
        assert ops.matmul_plan(535, 4096, 4096)[4] == plain
    # neighbours of the same step of rows take the height that is theirs; a plain entry does not speak for them
    size = {"rows": 352, "N": 5120, "K": 5120}
    ops.matmul_table([dict(size, kind="plain_round", own=32 + 7), dict(size, kind="plain", library=0)], clear=True)
    _forget_choices(ops)
    w = _rand((5120, 5120), torch.bfloat16, 33, scale=0.05)
    for M, height in ((330, 7), (340, 8)):
        ops.linear(_rand((M, 5120), torch.bfloat16, 34), w)
        assert ops.matmul_plan(M, 5120, 5120)[4] == 32 + height
    for entry in (dict(own=22), dict(own=18, splits=2), dict(own=42)):
        with pytest.raises(RuntimeError):
            ops.matmul_table([dict({"kind": "scaled", "rows": 208, "N": 4096, "K": 1024}, **entry)])


# long inner sizes of small weights, large weights that leave many CUs idle, and their neighbours on the other side of either line
@pytest.mark.parametrize("kind,M,N,K,own", [
    ("residual", 320, 1024, 8192, 8), ("residual", 320, 1024, 4864, 18), ("scaled", 640, 512, 16384, 8), ("scaled", 64, 1024, 8192, 8),
    ("scaled", 100, 1792, 5120, 17), ("scaled", 200, 768, 8192, 5), ("residual", 320, 2048, 4608, 8), ("residual", 320, 2048, 4096, 19), ("residual", 400, 896, 4864, 18),
    ("scaled_swiglu", 128, 22528, 4096, -1), ("scaled_swiglu", 128, 23552, 4096, 21), ("scaled", 128, 18432, 5120, -1),
    ("scaled", 97, 18432, 2048, 21), ("scaled", 97, 18432, 2112, -1), ("residual", 128, 24576, 4096, 8)])
def test_where_another_kernel_is_the_faster_one(rules_alone, kind, M, N, K, own):
    ops = rules_alone
    assert ops.matmul_fused_plan(kind, M, N, K)[0] == own
    x, w = _rand((M, K), torch.bfloat16, 91), _rand((N, K), torch.bfloat16, 92, scale=0.05)
    exact = x.double() @ w.double().T
    if kind == "residual":
        stream = torch.zeros(M, N, device="cuda")
        assert ops.linear_residual_norm(x, w, None, stream, torch.ones(N, device="cuda")) is not None
        got = stream
    else:
        sums = torch.full((1, ops.sums_stride(M)), float(K), device="cuda")
        got = ops.linear(x, w, unscaled=(sums, 0.0, K)) if kind == "scaled" else ops.linear_swiglu(x, w, unscaled=(sums, 0.0, K))
        if kind == "scaled_swiglu":
            exact = torch.nn.functional.silu(exact[:, ::2]) * exact[:, 1::2]
    torch.testing.assert_close(got.double(), exact, rtol=1.6e-2, atol=0.1)


def test_rows_off_sixteen_bytes_stay_the_few_row_kernels(monkeypatch):
    """32 rows that begin eight bytes off a multiple of sixteen: not a kernel's that copies them sixteen bytes at a time, the same bits."""
    ops = _ops()
    M, N, K = 32, 4096, 1024
    x, w = _rand((M, K), torch.bfloat16, 98), _rand((N, K), torch.bfloat16, 99, scale=0.05)
    tiled, sums = ops.tile_weight(w), torch.rand((64, M), generator=torch.Generator().manual_seed(97)).cuda() * 32.0
    more = dict(tiled=tiled, unscaled=(sums, 1e-5, K))
    flat = torch.empty(M * K + 4, dtype=torch.bfloat16, device="cuda")
    flat[4:] = x.view(-1)
    off, want, gated = flat[4:].view(M, K), ops.linear(x, w, **more), ops.linear_swiglu(x, w, **more)
    assert off.data_ptr() % 16 == 8

    def copies(*args):
        raise AssertionError("rows off sixteen bytes")

    monkeypatch.setattr(ops, "_tiles_scaled", copies)
    assert torch.equal(ops.linear(off, w, **more), want) and torch.equal(ops.linear_swiglu(off, w, **more), gated)
