"""Plain products of some hundred rows that one round of tiles covers, at the edges of the tiles and of the rule."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

HEIGHTS = 32       # `matmul_plan`'s number of such a tile, plus its height in units of 16 rows


# every height, rows and columns that end inside a tile, columns that no store of four takes, inner sizes of an odd
# number of stages, the least and the largest
@pytest.mark.parametrize("M,N,K,height", [(288, 4096, 4096, 5), (640, 2048, 4096, 5), (281, 4093, 2176, 5), (325, 4096, 4096, 6),
                                          (448, 4095, 2176, 7), (385, 4090, 5120, 7), (511, 4096, 3968, 8), (535, 4096, 4096, 9),
                                          (560, 4050, 4096, 9), (416, 5120, 5120, 9), (135, 8192, 1152, 5)])
def test_products_of_one_round(M, N, K, height):
    ops = _ops()
    x, w = _rand((M, K), torch.bfloat16, 31), _rand((N, K), torch.bfloat16, 32, scale=0.05)
    beyond = torch.full((M * N + 64,), 7.0, dtype=torch.bfloat16, device="cuda")
    got = ops.linear(x, w, out=beyond[:M * N].view(M, N))
    assert ops.matmul_plan(M, N, K)[4] == HEIGHTS + height
    exact = x.double() @ w.double().T
    # float32 sums of K exact products, and the rounding to bfloat16 (half a unit: 2^-9 of the value, 2^-8 with its ties)
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T) + 2.0 ** -8 * exact.abs()
    assert bool(((got.double() - exact).abs() <= bound).all())
    assert bool((beyond[M * N:] == 7.0).all())


@pytest.mark.parametrize("M,N,K", [(256, 4096, 4096), (641, 2048, 4096), (288, 4096, 4160), (535, 4096, 12288), (128, 8192, 2048)])
def test_sizes_that_stay_elsewhere(M, N, K):
    ops = _ops()
    x, w = _rand((M, K), torch.bfloat16, 33), _rand((N, K), torch.bfloat16, 34, scale=0.05)
    ops.linear(x, w)
    assert ops.matmul_plan(M, N, K)[4] < HEIGHTS


def test_misaligned_rows_and_a_product_in_float32_stay_elsewhere():
    ops = _ops()
    M, N, K = 300, 4096, 4096
    flat, w = _rand((M * K + 1,), torch.bfloat16, 35), _rand((N, K), torch.bfloat16, 36, scale=0.05)
    x = flat[1:].view(M, K)
    exact = x.double() @ w.double().T
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((ops.linear(x, w).double() - exact).abs() <= bound + 2.0 ** -8 * exact.abs()).all())
    assert bool(((ops.linear(x, w, out_dtype=torch.float32).double() - exact).abs() <= bound).all())
