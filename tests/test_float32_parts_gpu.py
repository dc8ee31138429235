"""float32 products with a weight that bfloat16 holds exactly, from its bfloat16 copy (`ops.narrow_weight`), at the edges
of their tiles, against float64."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def _weight(N, K, seed, scale=0.1):
    return _rand((N, K), torch.float32, seed, scale=scale).bfloat16().float()


# the few-row kernel (each of its row counts), every tile of the dispatch (32 x 16, 32 x 32, 32 x 64, 64 x 128), rows and
# columns that end inside a tile, inner sizes of one stage (three shares of K empty), of five (a share empty, one short) and of many; of one and of
# three where K is not shared out
@pytest.mark.parametrize("M,N,K", [(1, 1, 64), (4, 21, 512), (7, 130, 576), (16, 999, 1024), (17, 2, 64), (33, 1030, 320),
                                   (100, 1026, 192), (65, 2050, 1088), (130, 4094, 320), (257, 6146, 64), (1030, 3010, 448),
                                   (600, 2050, 64), (301, 4094, 192)])
def test_products_from_the_copy(M, N, K):
    ops = _ops()
    x, w = _rand((M, K), torch.float32, 81), _weight(N, K, 82)
    narrow = ops.narrow_weight(w)
    assert torch.equal(narrow.float(), w)
    got = ops.linear(x, w, narrow=narrow)
    want = x.double() @ w.double().T
    # at most K + K / 8 roundings of half a unit in the last place of the sum of the magnitudes, as for a chain of additions
    bound = 1.125 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - want).abs() <= bound).all())
    # no further off than the kernel on the float32 weight, by more than the two spread
    old = ops.linear(x, w)
    assert (got.double() - want).norm() <= 1.25 * (old.double() - want).norm()
    # a row's values depend neither on its neighbours nor on the tile that their number picks
    if M > 16:
        for part in (x[:17], x[M - 17:], x[:max(17, M // 3)]):
            first = part.storage_offset() // K
            assert torch.equal(ops.linear(part.contiguous(), w, narrow=narrow), got[first:first + part.shape[0]])
    # rows at odd addresses go by the float32 weight
    flat = torch.empty(M * K + 1, device="cuda")
    flat[1:] = x.view(-1)
    assert torch.equal(ops.linear(flat[1:].view(M, K), w, narrow=narrow), ops.linear(flat[1:].view(M, K), w))
    if N % 2 == 0:
        assert torch.equal(ops.linear_swiglu(x, w, narrow=narrow), ops.swiglu(got))
        assert torch.equal(ops.linear_swiglu(x, w, kind="gelu_erf", narrow=narrow), ops.gated_act(got, "gelu_erf"))


@pytest.mark.parametrize("M", [5, 40, 700])
def test_every_float32_number(M):
    """Infinities, NaN, zeros, the largest numbers and those whose lower bits bfloat16 has no exponent for."""
    ops = _ops()
    N, K = 2050, 320
    x, w = _rand((M, K), torch.float32, 83), _weight(N, K, 84)
    x[0, 5], x[1, 7], x[2, 300] = INF, -INF, NAN
    x[3] = torch.rand((K,), generator=torch.Generator().manual_seed(85)).cuda() * 2.0 ** -120
    x[4, ::2] = 0.0
    x[4, 1::2] *= 2.0 ** 120
    narrow = ops.narrow_weight(w)
    got, old = ops.linear(x, w, narrow=narrow), ops.linear(x, w)
    want = x.double() @ w.double().T
    for row in (0, 1, 2):
        assert torch.equal(got[row].nan_to_num(nan=7.0), old[row].nan_to_num(nan=7.0))
    bound = 1.125 * K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().T)
    assert bool(((got.double() - want).abs() <= bound)[3:].all())


def test_what_has_a_copy():
    ops = _ops()
    w = _weight(40, 128, 86)
    assert ops.narrow_weight(w) is not None
    for change in (0.1, INF, NAN):
        other = w.clone()
        other[39, 127] = change
        assert ops.narrow_weight(other) is None
    assert ops.narrow_weight(w.bfloat16()) is None and ops.narrow_weight(w.cpu()) is None
    assert ops.narrow_weight(w[:, :96].contiguous()) is None
    with pytest.raises(ValueError):
        ops.linear(_rand((3, 128), torch.float32, 87), w, narrow=ops.narrow_weight(w[:39]))


def test_copies_leave_room(monkeypatch):
    """A model's copies are made when everything is loaded and end where a quarter of what is free is theirs; the products of the
    matrices that have none are the float32 kernels', and no model has to have them."""
    from qwen3_from_scratch_amd.config import ModelConfig
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry, random_model
    from qwen3_from_scratch_amd.parts import linear

    config = ModelConfig.from_dict(dict(
        architectures=["Qwen3ForCausalLM"], vocab_size=512, hidden_size=256, hidden_act="silu", num_hidden_layers=2,
        max_position_embeddings=512, num_attention_heads=4, num_key_value_heads=2, head_dim=64, intermediate_size=512,
        rms_norm_eps=1e-6, rope_theta=1e6, tie_word_embeddings=False))
    first = 2 * (512 * 256 + 256 * 256)              # bytes of the copies of the first layer's attention
    held, logits = [], []
    for free, tiled in ((1 << 40, True), (4 * first, True), (0, True), (1 << 40, False)):
        asked = []
        monkeypatch.setattr(linear, "free_memory", lambda device: asked.append(torch.cuda.memory_allocated()) or free)
        model = random_model(config, dtype="float32", device="cuda:0", seed=5, tiled_weights=tiled)
        matrices = [m for m in linear._matrices(list(model.parts()), set())]
        held.append([m.narrow is not None for m in matrices])
        assert len(asked) == tiled and all(at >= sum(4 * m.weight.numel() for m in matrices) for at in asked)
        logits.append(ModelRunner(model, 16, 32, max_requests=2).step([StepEntry("a", list(range(40)), [39])]).clone())
    assert held == [[True] * 9, [True] * 2 + [False] * 7, [False] * 9, [False] * 9]
    for other in logits[1:]:
        torch.testing.assert_close(other, logits[0], rtol=1e-4, atol=1e-5)
    assert torch.equal(logits[2], logits[3])
