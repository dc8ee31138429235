"""Attention with capped scores and a gate behind its results (a build of its own), against float64: results that one block finishes and
results that are merged out of several blocks' parts, of single tokens, of prompts and of both in one launch."""

import pytest
import torch

from test_kernels_gpu import _ops, _paged_case, _rand
from test_mixed_attention_gpu import _bound, _exact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Hq,Hkv,D,page", [(8, 2, 128, 16), (16, 8, 64, 32)])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("lens,parts,prompt_parts", [
    ([(1, 40), (1, 200), (1, 1)], False, False), ([(1, 700), (1, 2500), (1, 40)], True, False),      # single tokens, whole and in parts
    ([(100, 3000)], False, True), ([(33, 2100), (40, 40)], False, True),                             # prompts, keys in parts
    ([(200, 200), (130, 177)], False, False), ([(19, 300)], False, False),
    ([(1, 2500), (100, 3000), (1, 40)], True, True),                                                 # both, either merged
    ([(1, 60 * i + 1) for i in range(22)] + [(600, 611)], None, False)])
def test_results_leave_through_the_gate(Hq, Hkv, D, page, wide, lens, parts, prompt_parts):
    ops = _ops()
    q_lens, kv_lens = [q for q, _ in lens], [k for _, k in lens]
    longest = max([k for q, k in lens if q > 1] or [0])
    T, G = sum(q_lens), Hq // Hkv
    if parts is not None:
        assert (min(q_lens) * G <= 16 and ops._splits(len(lens), Hkv, max(kv_lens)) > 1) == parts
    if max(q_lens) > 1:
        lib = ops.library("attention_capped_gated")
        assert (lib.q3_paged_attention_prompt_splits(T, Hq, Hkv, longest) > 1) == prompt_parts
    q, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, len(lens), Hq, Hkv, D, page, q_lens, kv_lens, 70)
    gate = _rand((T, 3 + Hq * (D if wide else 1)), torch.float32, 71)[:, 2:-1]      # rows apart, off sixteen bytes
    sink = torch.randn(Hq, generator=torch.Generator().manual_seed(72)).cuda()
    options = dict(min_q_len=min(q_lens), max_kv_len_of_many=longest or None, softcap=12.0)
    for s in (None, sink):
        got = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5, sink=s, gate=gate, **options)
        want, size = _exact(q, kc, vc, bt, cu, kvl, D ** -0.5, s, 12.0)
        open_by = torch.sigmoid(gate.double())
        open_by = open_by if wide else open_by.repeat_interleave(D, dim=1)
        assert bool(((got.double() - want * open_by).abs() <= _bound(got, size * open_by)).all())
    # without a gate the other build serves, also right behind a call with one
    plain = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5, **options)
    want, size = _exact(q, kc, vc, bt, cu, kvl, D ** -0.5, None, 12.0)
    assert bool(((plain.double() - want).abs() <= _bound(plain, size)).all())
