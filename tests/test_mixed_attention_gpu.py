"""Attention of a step with sequences of few and of many rows: one launch for both kinds."""

import pytest
import torch

import torch_ops
from test_kernels_gpu import _ops, _paged_case

pytestmark = pytest.mark.gpu


def _lens(name):
    g = torch.Generator().manual_seed(31)
    some = torch.randint(1, 500, (200,), generator=g).tolist()
    return {
        # (rows, keys): prompts among decoding ones, rows at the line between the kinds (16 / G), one tile and a row more
        "among": [(1, 33), (65, 65), (1, 700), (2, 9), (4, 40), (5, 300), (129, 500), (1, 1)],
        # the last of more than a wavefront of sequences, and the sixty-fourth and sixty-fifth
        "many": [(1, n) for n in some[:63]] + [(40, 40), (70, 90)] + [(1, n) for n in some[63:120]] + [(33, 200)],
        # keys shared out for both kinds: a few requests and a portion over a long prefix
        "shared": [(1, 2500), (100, 3000), (1, 40)],
        # so many rows that the decoding ones come first
        "filled": [(1, 600)] * 5 + [(1200, 1300)] + [(1, 77)] * 3 + [(900, 900)],
        # sequences without rows, and as many short prompts as their rows allow
        "short": [(1, 5), (0, 40), (17, 17), (17, 64), (0, 1), (17, 30), (17, 17)],
    }[name]


@pytest.mark.parametrize("Hq,Hkv,D,page", [(8, 2, 128, 16), (16, 8, 128, 16), (3, 3, 64, 32), (16, 1, 64, 16)])
@pytest.mark.parametrize("name", ["among", "many", "shared", "filled", "short"])
@pytest.mark.parametrize("with_sink", [False, True])
def test_few_and_many_rows_in_one_launch(name, Hq, Hkv, D, page, with_sink):
    ops = _ops()
    lens = _lens(name)
    q_lens, kv_lens = [q for q, _ in lens], [k for _, k in lens]
    q, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, len(lens), Hq, Hkv, D, page, q_lens, kv_lens, 32)
    sink = torch.randn(Hq, generator=torch.Generator().manual_seed(33)).cuda() if with_sink else None
    got = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5, min_q_len=1,
                              max_kv_len_of_many=max(k for q, k in lens if q > 1), sink=sink)
    assert bool(got.isfinite().all())
    # each kind by itself has kernels of its own: the same sums in the same order where the keys are shared out alike
    G = Hq // Hkv
    for kind in (lambda n: 0 < n * G <= 16, lambda n: n * G > 16):
        at = [b for b, n in enumerate(q_lens) if kind(n)]
        rows = torch.cat([torch.arange(int(cu[b]), int(cu[b + 1])) for b in at]).cuda()
        counts = [q_lens[b] for b in at]
        few = counts[0] * G <= 16
        alone = ops.paged_attention(q[rows].contiguous(), Hq, kc, vc, bt[at].contiguous(),
                                    torch.tensor([0] + counts).cumsum(0).int().cuda(), kvl[at].contiguous(),
                                    max(counts) if few else max(q_lens), max(kv_lens), D ** -0.5, min_q_len=1 if few else min(counts),
                                    max_kv_len_of_many=max(k for q, k in lens if q > 1), sink=sink)
        # two bfloat16 results of the same float32 sums in other orders: a rounding of 2^-8 of the value, values of a softmax
        # over unit normals
        torch.testing.assert_close(got[rows].float(), alone.float(), rtol=2.0 ** -7, atol=2.0 ** -9)
    if sink is None:
        want = torch_ops.paged_attention(q.float(), Hq, kc.float(), vc.float(), bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5)
        torch.testing.assert_close(got.float(), want.float(), rtol=2e-2, atol=2e-2)
