"""All layers of a step of single tokens in one launch against the same layers run part by part."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(layers=3, **sizes):
    from qwen3_from_scratch_amd.config import ModelConfig
    from qwen3_from_scratch_amd.models.decoder import build_model
    from qwen3_from_scratch_amd.parts.base import Precision
    from qwen3_from_scratch_amd.weights import RandomWeights

    shape = dict(hidden_size=1024, num_attention_heads=16, num_key_value_heads=8, head_dim=128, intermediate_size=2048)
    config = ModelConfig.from_dict(dict(
        dict(shape, **sizes), architectures=["Qwen3ForCausalLM"], vocab_size=512, hidden_act="silu", num_hidden_layers=layers,
        max_position_embeddings=8192, rms_norm_eps=1e-6, rope_theta=1e6, tie_word_embeddings=False))
    model = build_model(config, Precision.named("bfloat16"), "cuda:0")
    model.load(RandomWeights(model.tensors(), seed=5, std=0.02, norm_jitter=0.1, generate_on="cuda:0"))
    return model


def _logits(model, lengths, steps, graphs=False, page=16, launch=True):
    """Per step the logits of a request of each length that decodes a token."""
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry

    g = torch.Generator().manual_seed(3)
    runner = ModelRunner(model, page, sum(n // page + 2 for n in lengths) + 1, max_requests=len(lengths), use_graphs=graphs)
    ids = [torch.randint(0, 512, (n + steps,), generator=g).tolist() for n in lengths]
    run = model.decode_run
    for i, n in enumerate(lengths):
        runner.step([StepEntry(i, ids[i][:n], [])])
    model.decode_run = run if launch else None
    try:
        return torch.stack([runner.step([StepEntry(i, [ids[i][n + s]], [0]) for i, n in enumerate(lengths)]).clone()
                            for s in range(steps)])
    finally:
        model.decode_run = run


# the fewest and the most rows and those around the ways they are asked for; contexts without old keys, of a tile's edges and of several
# splits; steps of K that are no multiple of a wavefront's sixteen; one key head and as many as heads; a page of 32
@pytest.mark.parametrize("rows,longest,sizes,page", [
    (1, 1, {}, 16), (1, 32, {}, 16), (1, 700, dict(intermediate_size=3072), 16), (2, 2100, dict(hidden_size=640, intermediate_size=1408), 16),
    (3, 65, dict(num_attention_heads=8, num_key_value_heads=1), 32), (4, 300, dict(num_attention_heads=4, num_key_value_heads=4), 16),
    (5, 97, dict(hidden_size=2560, intermediate_size=9728), 16), (8, 513, {}, 16), (9, 40, dict(hidden_size=256, intermediate_size=384, num_attention_heads=2, num_key_value_heads=1), 16),
    (16, 260, dict(intermediate_size=5120), 16), (17, 90, {}, 16), (24, 400, dict(intermediate_size=3072), 16),
    (32, 35, dict(hidden_size=384, num_attention_heads=6, num_key_value_heads=2, intermediate_size=640), 16)])
def test_against_the_parts(rows, longest, sizes, page):
    model = _model(**sizes)
    assert model.decode_run is not None
    lengths = [max(1, longest - 13 * i) for i in range(rows)]
    want = _logits(model, lengths, 3, page=page, launch=False)
    got = _logits(model, lengths, 3, page=page)
    # both round every product and row to bfloat16 (each some 0.008 off exact numbers over these layers), at sums in other orders
    assert (got - want).norm() <= 0.02 * want.norm()
    assert not torch.equal(got, want)                    # (it was another kernel)
    if rows in (1, 2, 3, 8, 16, 24):                        # (sizes that graphs are captured for: no row fills up)
        replayed = _logits(model, lengths, 3, page=page, graphs=True, launch=True)
        assert (replayed - want).norm() <= 0.02 * want.norm()


def test_any_number_of_blocks_gives_the_same_bits(monkeypatch):
    """Fewer blocks than there is work for, one alone, and more than find room at once, where those that are there go on by themselves."""
    from qwen3_from_scratch_amd.ops.layers import DecodeLayers

    model = _model()
    lengths = [400, 77, 1]
    want = _logits(model, lengths, 2)
    run = DecodeLayers.run
    for blocks, patience in ((1, 64), (7, 64), (100, 64), (300, 64), (300, 1)):
        monkeypatch.setattr(DecodeLayers, "run", lambda self, *args, **named: run(self, *args, **dict(named, blocks=blocks, patience=patience)))
        assert torch.equal(_logits(model, lengths, 2), want), blocks


def test_what_is_not_taken():
    from qwen3_from_scratch_amd import ops

    model = _model()
    native = model.decode_run.native
    rows = torch.zeros(33, 1024, device="cuda")
    caches = [(torch.zeros(4, 8, 16, 128, dtype=torch.bfloat16, device="cuda"), torch.zeros(4, 8, 128, 16, dtype=torch.bfloat16, device="cuda"))] * 3
    table, lens = torch.zeros(33, 4, dtype=torch.int32, device="cuda"), torch.ones(33, dtype=torch.int32, device="cuda")
    assert not native.run(rows, caches, table, lens, 1, None)                # more rows than there are registers for
    wide = _model(hidden_size=1152).decode_run.native
    assert not wide.run(torch.zeros(17, 1152, device="cuda"), caches, table, lens[:17], 1, None)      # or than it is the faster way for
    with pytest.raises(ops.OperandError):
        native.run(rows[:4], caches[:2], table, lens[:4], 1, None)
    with pytest.raises(ops.OperandError):
        native.run(rows[:4], caches, table, lens[:4], 65, None)              # longer than the block table
    assert _model(head_dim=64).decode_run is None
    for small in (dict(hidden_size=128), dict(intermediate_size=128), dict(num_attention_heads=1, num_key_value_heads=1)):
        assert _model(**small).decode_run is None        # (wavefronts without a step of K: their loads would start before the weights)
    layer = dict(native.layers[0], down_tiles=native.layers[0]["down_tiles"][:-1])
    sizes = dict(heads=16, kv_heads=8, dim=128, width=1024, inner=2048, qk_eps=1e-6, scale=1.0)
    assert type(native).of([native.layers[0]], window=0, **sizes) is not None
    assert type(native).of([native.layers[0]], window=8, **sizes) is None and type(native).of([layer], window=0, **sizes) is None
