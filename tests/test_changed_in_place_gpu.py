"""Weights of which something else was made when a model was loaded, changed in place afterwards: every step goes by what they are now,
prompts and single tokens, captured or not."""

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _model(dtype, kind="rglru"):
    from qwen3_from_scratch_amd.config.surasun_config import SurasunConfig
    from qwen3_from_scratch_amd.engine import random_model

    mixers = {"mamba2": dict(heads=4, vdim=32, state=32, groups=1, conv=4, norm_groups=1), "rglru": dict(width=128, blocks=4, conv=4)}
    config = SurasunConfig.from_dict({
        "architecture": "Surasun", "vocab": 200, "width": 128, "norm": {"eps": 1e-5}, "residual_mult": 1.0, "streams": 3,
        "layers": [{"type": k, "mixer": mixers[k], "mlp": {"kind": "dense", "ff": 128}} for k in (kind, "mamba2")]})
    return random_model(config, dtype=dtype, device=DEV, seed=3, std=0.06)


def _steps():
    from qwen3_from_scratch_amd.engine import StepEntry

    return [[StepEntry("a", list(range(80)), [79]), StepEntry("b", list(range(9)), [8])]] + [
        [StepEntry("a", [7 + i], [0]), StepEntry("b", [9 + i], [0])] for i in range(3)]


def _change(model, what):
    with torch.no_grad():
        if what == "tables":
            model.layers[0].block.tables[1][2].add_(torch.eye(3, device=DEV))
            model.layers[1].block.tables[2][1].mul_(-0.5)
        elif what == "another table":
            read, write, mix = model.layers[1].block.tables[1]
            model.layers[1].block.tables[1] = (read * torch.tensor([3.0, -1.0, 0.5], device=DEV), write, mix)
        elif what == "gates":
            model.layers[0].mixer.gate_weights.mul_(-2.0)             # numbers that bfloat16 holds
        else:
            model.layers[0].mixer.gate_weights.add_(0.01)             # numbers that it does not


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("what", ["tables", "another table", "gates", "other gates"])
def test_every_step_goes_by_what_is_there(dtype, what):
    from qwen3_from_scratch_amd.engine import ModelRunner
    from qwen3_from_scratch_amd.models.stream_sources import stream_plan

    def run(model, runner):
        logits = [runner.step(step).clone() for step in _steps()]
        for request in ("a", "b"):
            runner.finish(request)
        return torch.cat(logits)

    model = _model(dtype)
    assert model.stream_plan is not None and model.layers[0].mixer.narrow_gates is not None
    runner = ModelRunner(model, 16, 32, max_requests=2)
    before = run(model, runner)
    assert torch.equal(run(model, runner), before)
    _change(model, what)
    after = run(model, runner)
    # a model that was so from the start, in steps that no graph was captured for
    other = _model(dtype)
    _change(other, what)
    unit = other.layers[0].mixer
    unit.narrow_gates, unit._narrow_of = None, (None, 0)
    other.stream_plan = stream_plan(other)
    want = run(other, ModelRunner(other, 16, 32, max_requests=2, use_graphs=False))
    assert torch.equal(after, want)
    assert float((after - before).norm() / before.norm()) > 1e-3
    # and back
    undone = _model(dtype)
    with torch.no_grad():
        for mine, theirs in zip(model.layers, undone.layers):
            for q, tables in mine.block.tables.items():
                for t, s in zip(tables, theirs.block.tables[q]):
                    t.copy_(s)
        model.layers[0].mixer.gate_weights.copy_(undone.layers[0].mixer.gate_weights)
    assert torch.equal(run(model, runner), before)


def test_a_pass_in_a_capture():
    """It cannot bring copies up to date, and goes by the weights themselves."""
    from qwen3_from_scratch_amd.engine import ModelRunner

    model = _model("float32")
    runner = ModelRunner(model, 16, 32, max_requests=2, use_graphs=False)
    steps = _steps()
    for step in steps[:2]:
        runner.step(step)
    caught = {}
    forward = model.forward

    def spy(batch, cache):
        caught["batch"] = batch
        return forward(batch, cache)

    model.forward = spy
    kept = [t.clone() for t in runner.storage.states]
    runner.step(steps[2])
    for t, s in zip(runner.storage.states, kept):
        t.copy_(s)
    _change(model, "tables")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        captured = forward(caught["batch"], runner.storage)
    graph.replay()
    torch.cuda.synchronize()
    for t, s in zip(runner.storage.states, kept):
        t.copy_(s)
    eager = forward(caught["batch"], runner.storage)
    assert torch.allclose(captured, eager, rtol=1e-4, atol=1e-4)
