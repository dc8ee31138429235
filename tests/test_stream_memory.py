"""A residual kept as sublayers' results takes no more memory than its streams do."""

import pytest
import torch

from qwen3_from_scratch_amd.models.stream_sources import results_most


@pytest.mark.parametrize("streams,size", [(s, size) for s in range(2, 9) for size in (2, 4)])
def test_results_in_the_place_of_streams(streams, size):
    from qwen3_from_scratch_amd import ops

    n = results_most(streams, size)
    assert 1 <= n and n * size <= 4 * streams + size          # and the result that joins the streams next
    assert 1 + n + 2 <= ops.SOURCES_MOST                      # the embedding and a sublayer of two sides beside them


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,streams,kind,ff", [("bfloat16", 4, "mamba2", 512), ("bfloat16", 2, "mamba2", 512), ("float32", 4, "mamba2", 512),
                                                   ("bfloat16", 8, "rglru", 256), ("float32", 2, "rglru", 0)])
def test_a_long_prompt_of_a_deep_model(dtype, streams, kind, ff):
    from qwen3_from_scratch_amd.config.surasun_config import SurasunConfig
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry, random_model

    mixers = {"mamba2": dict(heads=8, vdim=32, state=32, groups=1, conv=4, norm_groups=1), "rglru": dict(width=256, blocks=8, conv=4)}
    config = SurasunConfig.from_dict({
        "architecture": "Surasun", "vocab": 100, "width": 256, "norm": {"eps": 1e-5}, "residual_mult": 1.0, "streams": streams,
        "layers": [{"type": kind, "mixer": mixers[kind], "mlp": {"kind": "dense", "ff": ff} if ff else None} for _ in range(16)]})
    model = random_model(config, dtype=dtype, device="cuda:0", seed=1)
    runner = ModelRunner(model, 16, 600, max_requests=1)
    plan, peaks = model.stream_plan, []
    assert plan is not None
    for model.stream_plan in (None, plan, None, plan):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        torch.cuda.reset_peak_memory_stats()
        runner.step([StepEntry("a", [i % 100 for i in range(8192)], [8191])])
        torch.cuda.synchronize()
        peaks.append(torch.cuda.max_memory_allocated() - before)
        runner.finish("a")
    assert peaks[3] <= 1.02 * peaks[2], peaks
