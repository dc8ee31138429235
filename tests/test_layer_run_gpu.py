"""Stretches of layers that run as one native call against the same layers run part by part."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(layers=5, dtype="bfloat16", head_dim=128, inner=2048, tiled=True, **mixer):
    from qwen3_from_scratch_amd.config import ModelConfig
    from qwen3_from_scratch_amd.models.decoder import build_model
    from qwen3_from_scratch_amd.parts.base import Precision
    from qwen3_from_scratch_amd.weights import RandomWeights

    config = ModelConfig.from_dict(dict(
        architectures=["Qwen3ForCausalLM"], vocab_size=512, hidden_size=1024, hidden_act="silu", num_hidden_layers=layers,
        max_position_embeddings=8192, num_attention_heads=16, num_key_value_heads=8, head_dim=head_dim,
        intermediate_size=inner, rms_norm_eps=1e-6, rope_theta=1e6, tie_word_embeddings=False))
    components = {"mixer": {"name": "attention", "kwargs": mixer}} if mixer else None
    model = build_model(config, Precision.named(dtype, tiled=tiled), "cuda:0", components=components)
    model.load(RandomWeights(model.tensors(), seed=5, std=0.02, norm_jitter=0.1, generate_on="cuda:0"))
    model.config = config
    return model


def _steps(seed, *steps):
    from qwen3_from_scratch_amd.engine import StepEntry

    g = torch.Generator().manual_seed(seed)
    return [[StepEntry(rid, torch.randint(0, 512, (n,), generator=g).tolist(), [n - 1]) for rid, n in step] for step in steps]


def _logits(model, steps, calls=None, page=16):
    from qwen3_from_scratch_amd.engine import ModelRunner

    runner = ModelRunner(model, page, 700, max_requests=8)
    out = []
    for entries in steps:
        if calls is not None:
            calls.append(0)
        out.append(runner.step(entries).clone())
    return out


# prompts alone (of 65 and of 640 rows too), a portion beside requests that decode, with prefixes long enough that keys are
# shared out (decoding ones and a portion), and a step of too many rows, which is not the native call's
STEPS = ((("a", 65),), (("b", 200), ("a", 1)), (("c", 640),), (("a", 3000),), (("a", 300), ("b", 1), ("c", 1)), (("d", 641),),
         (("a", 1), ("b", 2), ("c", 70)))


def test_the_same_bits(monkeypatch):
    from qwen3_from_scratch_amd.ops.layers import DecoderLayers

    model = _model()
    assert sorted(model.runs) == [0, 1, 2, 3] and len(set(map(id, model.runs.values()))) == 1
    steps = _steps(6, *STEPS)
    took = []
    run = DecoderLayers.run

    def counted(self, first, count, *args):
        done = run(self, first, count, *args)
        took[-1] = (first, count)
        assert done is not None
        return done

    monkeypatch.setattr(DecoderLayers, "run", counted)
    got = _logits(model, steps, took)
    # the first layer reads a norm's finished rows: the stretch begins behind it
    assert took == [(1, 3), (1, 3), (1, 3), 0, (1, 3), 0, (1, 3)]
    model.observer = lambda *args: None
    want = _logits(model, steps, took)
    assert took[7:] == [0] * 7
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_layers_that_are_not_taken():
    from qwen3_from_scratch_amd import ops

    assert not _model(dtype="float32", layers=3).runs
    model = _model(layers=3)
    native = model.runs[0].native
    assert [native.rows_fit(rows) for rows in (64, 65, 640, 641)] == [False, True, True, False]
    try:
        ops.matmul_kernels("library")                  # the residual's product is declined then
        assert not native.rows_fit(200)
    finally:
        ops.matmul_kernels("both")
    layer = dict(native.layers[0], down=native.layers[0]["down"][:, :-64])
    sizes = dict(heads=16, kv_heads=8, dim=128, width=1024, inner=2048, qk_eps=1e-6, scale=1.0, window=0)
    assert type(native).of([native.layers[0]], **sizes) is not None and type(native).of([layer], **sizes) is None
    with pytest.raises(ops.OperandError):
        rows = torch.zeros(70, 1024, device="cuda")
        native.run(0, 1, rows, rows, rows, [(rows, rows)], rows, rows, rows, rows, rows, 70, 70, 70, None, None)


def test_layers_that_the_matrix_cores_do_not_attend_for(monkeypatch):
    """A head size that they take at no page leaves no stretch; a page that they do not take is found out once a step."""
    from qwen3_from_scratch_amd.ops.layers import DecoderLayers

    assert not _model(layers=3, head_dim=96).runs
    model, asked, run = _model(), [], DecoderLayers.run
    monkeypatch.setattr(DecoderLayers, "run", lambda self, *args: asked.append(run(self, *args)) or asked[-1])
    steps = _steps(7, (("a", 200),), (("b", 90), ("a", 1)))
    got = _logits(model, steps, page=24)
    assert asked == [None, None]
    model.observer = lambda *args: None
    for a, b in zip(got, _logits(model, steps, page=24)):
        assert torch.equal(a, b)


def test_a_cache_that_gives_views_alone():
    """What a model asks of a cache is `view`."""
    model = _model()
    steps = _steps(8, (("a", 200),))
    want = _logits(model, steps)
    forward = model.forward

    class Views:
        def __init__(self, cache):
            self.view = cache.view

    model.forward = lambda batch, cache: forward(batch, Views(cache))
    assert torch.equal(_logits(model, steps)[0], want[0])


@pytest.mark.parametrize("inner", [True, False])
def test_a_product_that_declines_after_all(monkeypatch, inner):
    """The product into the stream is declined when the settings change between the question and the step (here: by a
    number of partial sums that is not the kernel's): its layer is finished by its parts, as it would have been without the stretch."""
    from qwen3_from_scratch_amd.ops import layers

    steps = _steps(9, (("a", 200),), (("b", 90), ("a", 1)))
    lib, asked, run = layers._matmul(), [], layers.DecoderLayers.run

    class Other:
        q3_tiles_scaled, q3_tiles_residual = lib.q3_tiles_scaled, lib.q3_tiles_residual

        @staticmethod
        def q3_tiles_residual_chunks(M, N, K):
            return lib.q3_tiles_residual_chunks(M, N, K) + (2048 == K if not inner else 4096 == K)

    model = _model(inner=4096)                   # (the attention's output product has 2,048 numbers a row)
    monkeypatch.setattr(layers, "_matmul", lambda: Other)
    monkeypatch.setattr(layers.DecoderLayers, "run", lambda self, *args: asked.append(run(self, *args)) or asked[-1])
    got = _logits(model, steps)
    assert len(asked) == 4 and all(isinstance(d, layers.Declined) and d.layer == 0 and d.of_attention != inner for d in asked)
    model.observer = lambda *args: None
    for a, b in zip(got, _logits(model, steps)):
        assert float((a - b).norm() / b.norm()) < 0.02       # another rounding of one product in bfloat16 a layer


@pytest.mark.parametrize("mixer", [dict(qk_norm=False), dict(window=90), dict(qk_norm=False, window=33, scale=0.1)])
def test_the_same_bits_without_norms_of_the_heads_and_behind_a_window(mixer):
    model = _model(**mixer)
    assert sorted(model.runs) == [0, 1, 2, 3]
    native = model.runs[0].native
    assert native.window == mixer.get("window", 0) and (native.layers[0]["q_norm"] is None) == (mixer.get("qk_norm") is False)
    steps = _steps(10, (("a", 65),), (("b", 200), ("a", 1)), (("a", 300), ("b", 1)))
    got = _logits(model, steps)
    model.observer = lambda *args: None
    for a, b in zip(got, _logits(model, steps)):
        assert torch.equal(a, b)


def test_matrices_held_once_leave_no_stretch():
    assert not _model(layers=3, tiled=False).runs
