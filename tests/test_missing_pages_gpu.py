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

