"""The float32 path's matrix-core kernels (products of more than 16 rows, attention over pages of a multiple of 16)
at the edges of their tiles, against float64."""

import pytest
import torch

from test_kernels_gpu import _ops, _paged_case, _rand

pytestmark = pytest.mark.gpu


# every tile size of the dispatch (32 x 32, 32 x 64, 64 x 64, 64 x 128), rows and columns that end inside a tile, inner
# sizes shorter than a stage, that end inside one, and of every number of stages from one to four
@pytest.mark.parametrize("M,N,K", [(17, 1, 4), (31, 33, 20), (32, 64, 128), (33, 130, 132), (100, 1027, 260), (70, 6150, 64),
                                   (129, 6146, 68), (500, 4098, 100), (1030, 8130, 36), (2050, 4100, 388)])
def test_linear_float32_many_rows(M, N, K):
    ops = _ops()
    x, w = _rand((M, K), torch.float32, 61), _rand((N, K), torch.float32, 62, scale=0.1)
    got = ops.linear(x, w)
    want = x.double() @ w.double().T
    # a chain of K additions: at most K roundings of half a unit in the last place of the sum of the magnitudes
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - want).abs() <= bound).all())
    # a row's values do not depend on its neighbours, nor on the tile size that their number picks; and the sums run in
    # the order of the kernel for odd addresses, with the same bits
    flat = torch.empty(M * K + 1, device="cuda")
    flat[1:] = x.view(-1)
    assert torch.equal(ops.linear(flat[1:].view(M, K), w), got)
    for part in (x[:17], x[M - 17:], x[:max(17, M // 3)]):
        first = part.storage_offset() // K
        assert torch.equal(ops.linear(part.contiguous(), w), got[first:first + part.shape[0]])


def test_linear_float32_odd_addresses():
    """Operands that do not begin at a multiple of 16 bytes take the kernel that reads them one by one."""
    ops = _ops()
    flat, w = _rand((40 * 64 + 1,), torch.float32, 63), _rand((50, 64), torch.float32, 64)
    x = flat[1:].view(40, 64)
    torch.testing.assert_close(ops.linear(x, w).double(), x.double() @ w.double().T, rtol=1e-5, atol=1e-5)


def _attention(ops, case, Hq, scale, **more):
    q, kc, vc, bt, cu, kvl = case
    lens = cu.diff().tolist()
    return ops.paged_attention(q, Hq, kc, vc, bt, cu, kvl, max(lens), int(kvl.max()), scale, **more)


def _want(case, Hq, scale, window=0, sink=None):
    """In float64, row by row."""
    q, kc, vc, bt, cu, kvl = (t.cpu() for t in case)
    T, _, D = q.shape
    Hkv, page = kc.shape[1], kc.shape[2]
    out = torch.zeros(T, Hq, D, dtype=torch.float64)
    for b in range(kvl.numel()):
        L, first, n = int(kvl[b]), int(cu[b]), int(cu[b + 1] - cu[b])
        pages = bt[b, :-(-L // page)].long()
        K = kc[pages].double().permute(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :L].repeat_interleave(Hq // Hkv, 0)
        V = vc[pages].double().permute(1, 0, 3, 2).reshape(Hkv, -1, D)[:, :L].repeat_interleave(Hq // Hkv, 0)
        for i in range(n):
            end = L - n + i + 1
            start = max(0, end - window) if window else 0
            s = (K[:, start:end] @ q[first + i].double()[:, :, None])[..., 0] * scale
            if sink is not None:
                s = torch.cat((s, sink.cpu().double()[:, None]), dim=1)
            p = torch.softmax(s, dim=1)[:, :end - start]
            out[first + i] = (p[:, None, :] @ V[:, start:end])[:, 0]
    return out.view(T, Hq * D).cuda()


@pytest.mark.parametrize("Hq,Hkv,D,page", [(3, 3, 16, 16), (10, 2, 32, 48), (16, 1, 64, 16), (4, 2, 128, 32), (18, 2, 128, 64)])
@pytest.mark.parametrize("window,with_sink", [(0, False), (0, True), (23, False), (130, True)])
def test_attention_float32(Hq, Hkv, D, page, window, with_sink):
    """Sequences of one key, of one tile and a key more, of fewer tiles than wavefronts and of more, with single rows,
    rows that end inside a block, and NaN wherever no row may look."""
    ops = _ops()
    q_lens, kv_lens = [1, 16, 1, 5, 37, 1], [1, 16, 17, 129, 150, 600]
    case = _paged_case(torch.float32, 6, Hq, Hkv, D, page, q_lens, kv_lens, 71)
    q, kc, vc, bt, cu, kvl = case
    owned = torch.zeros(kc.shape[0], page, dtype=torch.bool)
    for b, L in enumerate(kv_lens):
        for j in range(L):
            owned[int(bt[b, j // page]), j % page] = True
    kc.transpose(1, 2)[~owned] = float("nan")
    vc.permute(0, 3, 1, 2)[~owned] = float("nan")
    sink = _rand((Hq,), torch.float32, 72) if with_sink else None
    scale = D ** -0.5
    got = _attention(ops, case, Hq, scale, window=window, sink=sink)
    torch.testing.assert_close(got.double(), _want(case, Hq, scale, window, sink), rtol=1e-4, atol=2e-5)
    # the last sequence but one again, its rows one at a time: the sums are the same
    first = sum(q_lens[:4])
    for i in (0, 1, 15, 36):
        one = (q[first + i:first + i + 1], kc, vc, bt[4:5], torch.tensor([0, 1], dtype=torch.int32).cuda(),
               torch.tensor([150 - 37 + i + 1], dtype=torch.int32).cuda())
        assert torch.equal(_attention(ops, one, Hq, scale, window=window, sink=sink)[0], got[first + i])


@pytest.mark.parametrize("L,at", [(1, 0), (16, 15), (17, 16), (33, 32), (200, 100), (129, 128)])
def test_attention_float32_keeps_a_nan(L, at):
    """A key of NaN is seen in the result, also where it is the only key of its tile and no wavefront has another; a row
    before it does not look."""
    ops = _ops()
    q, kc, vc, bt, cu, kvl = _paged_case(torch.float32, 1, 4, 2, 64, 16, [min(2, L)], [L], 73)
    kc[int(bt[0, at // 16]), :, at % 16] = float("nan")
    got = _attention(ops, (q, kc, vc, bt, cu, kvl), 4, 0.125)
    assert bool(got[-1].isnan().all())
    assert L == 1 or bool(got[0].isnan().all()) == (at < L - 1)
