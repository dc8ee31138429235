"""Every way in which a step's prompts go over blocks (rows of a block, the order beside decoding requests, sixteen rows a block), each
asked for by a step that is seen to take it, against float64."""

import pytest
import torch

from test_kernels_gpu import _ops, _paged_case
from test_mixed_attention_gpu import _bound, _exact
from test_prompt_plan_host import _plan

pytestmark = pytest.mark.gpu

DECODING = [(1, 15 * i + 1) for i in range(23)]


@pytest.mark.parametrize("cap", [0.0, 12.0])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("Hq,Hkv,lens,rows,first,brief", [
    (16, 8, [(300, 311)], 32, None, False), (8, 8, [(20, 20)] * 62 + [(17, 40), (1, 3)], 32, None, False),
    (16, 8, [(700, 733), (690, 690), (17, 1200)], 64, None, False), (6, 2, [(1500, 1500), (1501, 1533)], 64, None, False),
    (16, 8, [(2500, 2517)], 128, None, False), (32, 8, [(70, 75)] * 16, 128, None, False), (12, 4, [(65, 65), (33, 300)], None, None, True),
    # beside decoding requests: prompts first, then those first that decode
    (16, 8, DECODING + [(300, 300)], 32, True, False), (16, 8, DECODING + [(600, 633)], 64, True, False),
    (16, 8, DECODING + [(1160, 1160)], 128, True, False),
    (16, 8, [(1, 1600)] + DECODING + [(300, 300)], 32, False, False), (16, 8, [(1, 3200)] + DECODING + [(600, 633)], 64, False, False),
    (16, 8, [(1, 6000)] + DECODING + [(1160, 1160)], 128, False, False), (32, 8, [(1, 700)] + [(130, 130)] * 14, 128, False, False),
    (16, 8, [(1, 150)] * 36 + [(20, 820)], None, None, True)])
def test_against_64_bits(Hq, Hkv, lens, rows, first, brief, D, cap):
    ops = _ops()
    q_lens, kv_lens = [q for q, _ in lens], [k for _, k in lens]
    plan = _plan((Hq, Hkv), q_lens, kv_lens)
    assert plan[2] == brief
    if not brief:
        G = Hq // Hkv
        assert plan[0] in (rows, rows // G * G) and (first is None or plan[1] == first) and plan[3] == 1
    q, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, len(lens), Hq, Hkv, D, 16, q_lens, kv_lens, 91)
    sink = torch.randn(Hq, generator=torch.Generator().manual_seed(92)).cuda()
    got = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5, min_q_len=min(q_lens),
                              max_kv_len_of_many=max(k for n, k in lens if n > 1), sink=sink, softcap=cap)
    want, size = _exact(q, kc, vc, bt, cu, kvl, D ** -0.5, sink, cap)
    assert bool(((got.double() - want).abs() <= _bound(got, size)).all())
