"""The edges of the kernels that keep a whole row, part, tile or state in registers: the smallest and largest rows that
they take and the next that they leave to the general kernels, rows that do not begin on sixteen bytes, remainders of
tiles, against the plain PyTorch twins. Tolerances are those of the general kernels' tests: sums of float32 products
in another order, one rounding to the result's type."""

import pytest
import torch

import torch_ops as twin
from qwen3_from_scratch_amd import ops
from test_surasun_kernels_gpu import DEV, DTYPES, _close, _gen, _rand, _step, _tol

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("S", [2, 4])
@pytest.mark.parametrize("W,off", [(4, 0), (252, 0), (260, 4), (260, 1), (4096, 0), (4100, 0)])
def test_hyper_norm_rows(dtype, S, W, off):
    g = _gen(S * W + off)
    T = 3
    x, weight, read, write, mix = _rand(g, T, S, W), _rand(g, W), _rand(g, S), _rand(g, S), _rand(g, S, S)
    delta = _rand(g, T * W + off, dtype=dtype)[off:].view(T, W)
    rows = torch.tensor([2, 0, 2, 1], dtype=torch.int32, device=DEV)
    for kwargs in (dict(), dict(read=read, delta=delta, mix=mix, write=write), dict(delta=delta, mix=mix, write=write, rows=rows)):
        a, b = x.clone(), x.clone()
        _close(ops.hyper_norm(a, weight, 1e-5, dtype, **kwargs), twin.hyper_norm(b, weight, 1e-5, dtype, **kwargs), _tol(dtype))
        _close(a, b, 1e-5)
    a, b = x.clone(), x.clone()
    assert ops.hyper_norm(a, None, 0.0, dtype, delta=delta, mix=mix, write=write) is None
    twin.hyper_norm(b, None, 0.0, dtype, delta=delta, mix=mix, write=write)
    _close(a, b, 1e-5)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,groups,off", [(4, 1, 0), (504, 2, 0), (520, 2, 4), (260, 1, 1), (4096, 1, 0), (8192, 2, 8), (4100, 1, 0)])
def test_gated_rmsnorm_rows(dtype, n, groups, off):
    g = _gen(n + off)
    y, weight = _rand(g, 3, n), _rand(g, n)
    gate = _rand(g, 3, n + 12, dtype=dtype)[:, off:off + n]
    _close(ops.gated_rmsnorm(y, gate, weight, groups, 1e-6, dtype), twin.gated_rmsnorm(y, gate, weight, groups, 1e-6, dtype),
           _tol(dtype))


@pytest.mark.parametrize("T,width,blocks", [(1, 64, 1), (17, 60, 2), (16, 1536, 1), (48, 2048, 8), (49, 2048, 8), (65, 2048, 2),
                                            (1970, 50, 2), (130, 1020, 15), (70, 3070, 2)])
def test_block_gates_both_ways(T, width, blocks):
    g = _gen(T + width)
    bw = width // blocks
    u, weights, biases = _rand(g, T, width), _rand(g, 2, blocks, bw, bw, scale=bw ** -0.5), _rand(g, 2, blocks, bw)
    z = torch.stack([u.double().view(T, blocks, bw)[:, b] @ weights[:, b].double() for b in range(blocks)], 2)
    want = torch.sigmoid(z + biases.double()[:, None]).reshape(2, T, width)
    # a sigmoid's slope is at most 1/4: a quarter of the error of a float32 sum of 1,536 products, whose partial sums are
    # of size 1 and drift by sqrt(1536) halves of 2^-23 (0.6e-6 in all); a few times that
    assert float((ops.block_gates(u, weights, biases).double() - want).abs().max()) < 4e-6
    aside = torch.empty(T * width + 1, device=DEV)[1:].view(T, width).copy_(u)      # rows that begin on four bytes
    assert float((ops.block_gates(aside, weights, biases).double() - want).abs().max()) < 4e-6


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,P,N,G,lengths", [(2, 64, 64, 1, [64, 65]), (2, 62, 65, 2, [127, 1]), (3, 68, 132, 1, [70, 63]),
                                             (1, 3, 1, 1, [66]), (2, 130, 256, 2, [129])])
def test_chunks_of_whole_and_broken_rows(dtype, H, P, N, G, lengths):
    """Keys of up to 64, 128 and 256 numbers, rows read four numbers at a time and one by one, chunks of one row."""
    g = _gen(H * P + N)
    T = sum(lengths)
    xbc, dt = _rand(g, T, H * P + 2 * G * N, dtype=dtype), _rand(g, T, H, dtype=dtype)
    dt_bias, a_log, skip = _rand(g, H), _rand(g, H, scale=0.5), _rand(g, H)
    cu, _, slots = _step(lengths, [1, 0][:len(lengths)])
    full = _rand(g, 2, H * N * P, scale=0.3)
    a, b = full.clone(), full.clone()
    assert max(lengths) >= ops.CHUNKED_FROM
    got = ops.mamba2_scan(xbc, dt, dt_bias, a_log, skip, a, slots, cu, H, P, N, G, max_q_len=max(lengths))
    _close(got, twin.mamba2_scan(xbc, dt, dt_bias, a_log, skip, b, slots, cu, H, P, N, G), 3e-5)
    _close(a, b, 3e-5)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,width,off", [(1, 1, 0), (16, 64, 0), (33, 68, 0), (64, 62, 0), (65, 130, 3), (128, 64, 2), (256, 256, 4)])
@pytest.mark.parametrize("lengths", [[1, 1], [8, 3]])
def test_state_walked_row_by_row(dtype, rows, width, off, lengths):
    """Sequences of one token and of several, states of rows and widths around the kernel's 16 EACH rows and 64 columns,
    on sixteen bytes or not."""
    g = _gen(rows * width + off)
    T, H = sum(lengths), 2
    cu, _, slots = _step(lengths, [2, 0])
    full = _rand(g, 3, H * rows * width + off, scale=0.3)
    xbc, dt = _rand(g, T, H * width + 2 * rows, dtype=dtype), _rand(g, T, H, dtype=dtype)
    dt_bias, a_log, skip = _rand(g, H), _rand(g, H, scale=0.5), _rand(g, H)
    a, b = full.clone(), full.clone()
    got = ops.mamba2_scan(xbc, dt, dt_bias, a_log, skip, a[:, off:], slots, cu, H, width, rows, 1, max_q_len=max(lengths))
    _close(got, twin.mamba2_scan(xbc, dt, dt_bias, a_log, skip, b[:, off:], slots, cu, H, width, rows, 1), 3e-5)
    _close(a, b, 3e-5)


@pytest.mark.parametrize("rows", [1, 16, 20, 32, 48, 66, 130])
def test_state_walked_with_an_infinite_input(rows):
    """An infinity in one column stays there, and one: rows that fill a state up to 16 EACH make no NaN of it."""
    H, P = 2, 8
    xbc, zero = torch.ones(2, H * P + 2 * rows, device=DEV), torch.zeros(H, device=DEV)
    xbc[0, 3] = float("inf")
    cu, _, slots = _step([2], [0])
    a, b = torch.zeros(1, H * rows * P, device=DEV), torch.zeros(1, H * rows * P, device=DEV)
    args = (xbc, torch.zeros(2, H, device=DEV), zero, zero, zero + 1)
    got = ops.mamba2_scan(*args, a, slots, cu, H, P, rows, 1, max_q_len=2)
    want = twin.mamba2_scan(*args, b, slots, cu, H, P, rows, 1)
    assert bool(want[:, 3].isinf().all()) and torch.equal(got.isinf(), want.isinf()) and not bool(got.isnan().any())
    torch.testing.assert_close(got[want.isfinite()], want[want.isfinite()], rtol=1e-5, atol=0)
    assert torch.equal(a.isinf(), b.isinf())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("C,taps,lengths", [(8, 4, [256]), (520, 4, [1, 2, 255]), (512, 4, [263, 1]), (520, 8, [259]), (1024, 1, [256])])
def test_causal_conv_tiles(dtype, C, taps, lengths):
    """Tiles of eight rows whole and broken, of one sequence and of two, the exact taps and any number."""
    g = _gen(C + taps)
    x = _rand(g, sum(lengths), C, dtype=dtype)
    weight, bias, add = _rand(g, C, taps), _rand(g, C), _rand(g, C)
    cu, seq, slots = _step(lengths, [4, 0, 2][:len(lengths)])
    full = _rand(g, 5, max(1, (taps - 1) * C))
    for in_bias in (None, add):
        a, b = full.clone(), full.clone()
        state_a, state_b = a[:, :(taps - 1) * C], b[:, :(taps - 1) * C]
        _close(ops.causal_conv(x, weight, bias, state_a, slots, cu, seq, "silu", dtype, in_bias, max_q_len=max(lengths)),
               twin.causal_conv(x, weight, bias, state_b, slots, cu, seq, "silu", dtype, in_bias), _tol(dtype))
        _close(a, b, 1e-6)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("H,G,dim,vdim,half,off", [(2, 1, 2, 1, 1, 0), (30, 2, 128, 128, 32, 0), (32, 2, 128, 64, 64, 0), (4, 4, 66, 512, 16, 2),
                                                   (4, 4, 64, 516, 0, 0), (4, 2, 64, 64, 16, 1)])
@pytest.mark.parametrize("transposed", [False, True])
def test_capped_preparation_rows(dtype, H, G, dim, vdim, half, off, transposed):
    """Rows that the registers hold (up to 4,096 numbers of q and k, 2,048 of v) and the next larger, on eight bytes or
    not, a page that is missing, no cache."""
    g = _gen(H * dim + vdim + off)
    T, page = 5, 16
    n = H * dim + G * dim + G * vdim
    rows = _rand(g, T, n + off + n % 2)[:, off:off + n]
    bias, qw, kw = _rand(g, n), _rand(g, H * dim), _rand(g, G * dim)
    inv_freq = torch.rand(half, generator=g).to(DEV) if half else None
    as_int = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    positions, seq, table = as_int([0, 17, 40, 3, 15]), as_int([0, 0, 0, 1, 1]), as_int([[2, 0, 3], [-1, 1, 1]])
    def caches():
        shape = (4, G, vdim, page) if transposed else (4, G, page, vdim)
        return torch.zeros(4, G, page, dim, dtype=dtype, device=DEV), torch.zeros(shape, dtype=dtype, device=DEV)
    for b in (bias, None):
        mine, other = caches(), caches()
        args = (rows, b, H, G, dim, vdim, qw, kw, 1e-6, inv_freq, positions, seq, dtype)
        live = [0, 1, 2]        # (the twin takes no missing page: the second sequence's tokens only there)
        got = ops.softcap_prepare(*args, table, *mine, values_transposed=transposed)
        want = twin.softcap_prepare(rows[live], b, H, G, dim, vdim, qw, kw, 1e-6, inv_freq, positions[live], seq[live], dtype, table,
                                    *other, values_transposed=transposed)
        _close(got[live], want, _tol(dtype))
        for x, y in zip(mine, other):
            _close(x, y, _tol(dtype))
        _close(ops.softcap_prepare(*args), twin.softcap_prepare(*args), _tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("W,off", [(4, 0), (260, 0), (4100, 0), (260, 1), (6, 0)])
def test_embed_streams_rows(dtype, W, off):
    table = _rand(_gen(W), 3 * W + off, dtype=dtype)[off:].view(3, W)
    ids = torch.tensor([2, -1, 0, 3], dtype=torch.int32, device=DEV)      # (outside the table: zeros)
    got = ops.embed_streams(ids, table, 3)
    for t, row in enumerate((table[2].float(), torch.zeros(W, device=DEV), table[0].float(), torch.zeros(W, device=DEV))):
        assert all(bool(torch.equal(got[t, s], row)) for s in range(3))
