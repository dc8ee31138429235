"""Attention of a step with sequences of few and of many rows: one launch for both kinds."""

import pytest
import torch

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
        # so few rows in all that both kinds go by blocks of sixteen: their last ones short, keys of one tile and of many
        "few": [(1, 33), (18, 18), (19, 200), (1, 64), (33, 300)],
        # sequences without rows, and as many short prompts as their rows allow
        "short": [(1, 5), (0, 40), (17, 17), (17, 64), (0, 1), (17, 30), (17, 17)],
    }[name]


def _exact(q, kc, vc, bt, cu, kvl, scale, sink, cap, window=0):
    """The attention in float64, and of every result the sum of the magnitudes that it adds."""
    Hq, Hkv, page = q.shape[1], kc.shape[1], kc.shape[2]
    result, size = [], []
    for b, L in enumerate(kvl.tolist()):
        rows = q[int(cu[b]):int(cu[b + 1])].double()
        n, pages = rows.shape[0], bt[b, :-(-L // page)].long()
        k = kc[pages].double().permute(1, 0, 2, 3).flatten(1, 2)[:, :L].repeat_interleave(Hq // Hkv, dim=0)
        v = vc[pages].double().permute(1, 0, 3, 2).flatten(1, 2)[:, :L].repeat_interleave(Hq // Hkv, dim=0)
        s = torch.matmul(rows.transpose(0, 1), k.transpose(1, 2).contiguous()) * scale
        s = cap * torch.tanh(s / cap) if cap else s
        behind = torch.arange(L - n, L, device="cuda")[:, None] - torch.arange(L, device="cuda")
        s = s.masked_fill((behind < 0) | (behind >= (window or L)), float("-inf"))
        if sink is not None:
            s = torch.cat((s, sink.double()[:, None, None].expand(Hq, n, 1)), dim=2)
        w = torch.softmax(s, dim=2)[:, :, :L]
        result.append(torch.matmul(w, v).transpose(0, 1).flatten(1))
        size.append(torch.matmul(w, v.abs()).transpose(0, 1).flatten(1))
    return torch.cat(result), torch.cat(size)


def _bound(got, size):
    """A bfloat16 result (eight significant bits: half a unit is 2^-8 of a number at most) is off by its own rounding and by that of
    the probabilities in the second product, 2^-8 of the sum of the magnitudes it adds; the rest, float32, is far below."""
    return 2.0 ** -8 * (size + got.double().abs()) * 1.05 + 1e-5


@pytest.mark.parametrize("Hq,Hkv,D,page", [(8, 2, 128, 16), (16, 8, 128, 16), (3, 3, 64, 32), (16, 1, 64, 16)])
@pytest.mark.parametrize("name", ["among", "many", "shared", "filled", "few", "short"])
@pytest.mark.parametrize("with_sink", [False, True])
@pytest.mark.parametrize("cap", [0.0, 12.0])             # (capped scores: a build of their own)
def test_few_and_many_rows_in_one_launch(name, Hq, Hkv, D, page, with_sink, cap):
    ops = _ops()
    lens = _lens(name)
    q_lens, kv_lens = [q for q, _ in lens], [k for _, k in lens]
    q, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, len(lens), Hq, Hkv, D, page, q_lens, kv_lens, 32)
    sink = torch.randn(Hq, generator=torch.Generator().manual_seed(33)).cuda() if with_sink else None
    got = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5, min_q_len=1,
                              max_kv_len_of_many=max(k for q, k in lens if q > 1), sink=sink, softcap=cap)
    assert bool(got.isfinite().all())
    want, size = _exact(q, kc, vc, bt, cu, kvl, D ** -0.5, sink, cap)
    bound = _bound(got, size)
    assert bool(((got.double() - want).abs() <= bound).all())
    # each kind by itself, in kernels of its own
    G = Hq // Hkv
    for kind in (lambda n: 0 < n * G <= 16, lambda n: n * G > 16):
        at = [b for b, n in enumerate(q_lens) if kind(n)]
        rows = torch.cat([torch.arange(int(cu[b]), int(cu[b + 1])) for b in at]).cuda()
        counts = [q_lens[b] for b in at]
        alone = ops.paged_attention(q[rows].contiguous(), Hq, kc, vc, bt[at].contiguous(),
                                    torch.tensor([0] + counts).cumsum(0).int().cuda(), kvl[at].contiguous(), max(counts),
                                    max(kv_lens), D ** -0.5, min_q_len=min(counts),
                                    max_kv_len_of_many=max(k for q, k in lens if q > 1), sink=sink, softcap=cap)
        assert bool(((got[rows].double() - alone.double()).abs() <= 2 * bound[rows]).all())


@pytest.mark.parametrize("Hq,Hkv,D,page", [(8, 2, 128, 16), (16, 8, 128, 16), (3, 3, 64, 32), (16, 1, 64, 16)])
@pytest.mark.parametrize("lens", [[(17, 1984)], [(40, 1900), (17, 17), (20, 1000)], [(33, 1970), (21, 1500)]])
@pytest.mark.parametrize("cap", [0.0, 12.0])
def test_few_rows_over_many_keys(Hq, Hkv, D, page, lens, cap):
    """Blocks of sixteen rows over as many keys as no block of them shares with another."""
    ops = _ops()
    q_lens, kv_lens = [q for q, _ in lens], [k for _, k in lens]
    assert ops.library("attention").q3_paged_attention_prompt_splits(sum(q_lens), Hq, Hkv, max(kv_lens)) == 1
    q, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, len(lens), Hq, Hkv, D, page, q_lens, kv_lens, 34)
    got = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5, min_q_len=min(q_lens), softcap=cap)
    want, size = _exact(q, kc, vc, bt, cu, kvl, D ** -0.5, None, cap)
    assert bool(((got.double() - want).abs() <= _bound(got, size)).all())


# Blocks of 32, 64 and 128 rows, whose wavefronts share the keys or do not: rows and keys at the edges of tiles and of their halves (the first row of a
# prompt sees no key of the second), keys in parts, a window, a group that does not divide the rows; the last two beside decoding ones
@pytest.mark.parametrize("Hq,Hkv,D,page,lens,window", [
    (8, 2, 128, 16, [(200, 200), (17, 33), (130, 177), (129, 1031)], 0), (8, 2, 64, 16, [(300, 300), (95, 128)], 0),
    (12, 4, 128, 32, [(260, 260), (100, 640)], 0), (16, 2, 128, 16, [(150, 3300)], 0), (8, 2, 128, 64, [(150, 4100), (40, 40)], 0),
    (8, 2, 128, 16, [(200, 260), (130, 177)], 40), (8, 8, 64, 16, [(1290, 1300), (1250, 1250)], 0), (6, 2, 128, 16, [(1500, 1500), (1501, 1533)], 0),
    (8, 8, 128, 16, [(1100, 1100), (1111, 1130)], 300), (8, 8, 64, 16, [(2410, 2433), (2400, 2400)], 0),
    (16, 8, 128, 16, [(1, 50 * i + 1) for i in range(16)] + [(600, 611)], 0), (16, 8, 64, 16, [(1, 30 * i + 1) for i in range(17)] + [(1300, 1300)], 0)])
@pytest.mark.parametrize("cap", [0.0, 12.0])
def test_rows_of_a_block(Hq, Hkv, D, page, lens, window, cap):
    ops = _ops()
    q_lens, kv_lens = [q for q, _ in lens], [k for _, k in lens]
    q, kc, vc, bt, cu, kvl = _paged_case(torch.bfloat16, len(lens), Hq, Hkv, D, page, q_lens, kv_lens, 35)
    sink = torch.randn(Hq, generator=torch.Generator().manual_seed(36)).cuda()
    got = ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(q_lens), max(kv_lens), D ** -0.5, window=window, min_q_len=min(q_lens),
                              max_kv_len_of_many=max(k for q, k in lens if q > 1), sink=sink, softcap=cap)
    want, size = _exact(q, kc, vc, bt, cu, kvl, D ** -0.5, sink, cap, window)
    assert bool(((got.double() - want).abs() <= _bound(got, size)).all())
