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
