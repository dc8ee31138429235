"""The gate and up product with its activation in one round of blocks: only while nobody has said which kernel the plain product of its
size is to go to."""

import pytest
import torch

from qwen3_from_scratch_amd import ops

SIZE = (535, 24576, 4096)


@pytest.fixture
def table():
    """The package's table, put back behind the test."""
    yield
    ops.matmul_tuner(False)
    ops.matmul_kernels("both")
    ops.matmul_table([], clear=True)
    ops._table_loaded = False
    ops._matmul()


def _entry(rows=SIZE[0], **choice):
    return dict(kind=ops.matmul_plain_kind(rows, SIZE[1], SIZE[2]), rows=ops.matmul_rows_key("plain", rows), N=SIZE[1], K=SIZE[2], out="bfloat16", **choice)


def test_who_decides(table):
    serves = ops._matmul().q3_wide_swiglu_serves
    assert serves(*SIZE) and not serves(512, *SIZE[1:])          # with the package's entries in
    ops.matmul_tuner(True)
    assert not serves(*SIZE)
    ops.matmul_tuner(False)
    for which in ("library", "own"):
        ops.matmul_kernels(which)
        assert not serves(*SIZE)
    ops.matmul_kernels("both")
    assert serves(*SIZE)
    ops.matmul_table([dict(_entry(library=1), N=4096)])
    assert serves(*SIZE)
    ops.matmul_table([_entry(library=1)])
    assert not serves(*SIZE) and not serves(520, *SIZE[1:]) and serves(570, *SIZE[1:])      # (rows 513 to 544 share an entry)
    ops.matmul_table([], clear=True)
    assert serves(*SIZE)


@pytest.mark.gpu
def test_an_entry_is_gone_by(table):
    M, N, K = SIZE
    x = torch.randn(M, K, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    w = (torch.randn(N, K, generator=torch.Generator().manual_seed(2)) * 0.05).bfloat16().cuda()
    ops.matmul_kernels("library")
    ops.matmul_kernels("both")                                   # (sizes that other tests have met choose anew)
    inside = ops.linear_swiglu(x, w)
    assert ops.matmul_plan(M, N, K) is None                      # no plain product has run
    ops.matmul_table([_entry(own=3, splits=1)])
    after = ops.linear_swiglu(x, w)
    assert ops.matmul_plan(M, N, K)[4] == 3
    assert torch.equal(after, ops.swiglu(ops.linear(x, w)))
    torch.testing.assert_close(after.float(), inside.float(), rtol=3.2e-2, atol=2e-2)
