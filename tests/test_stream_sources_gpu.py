"""A residual in several streams kept as the sums that its streams are: the kernels against float64, and a model's logits
against the same model with its streams in memory, short of, at and past the number of sublayers where the two change over."""

import pytest
import torch

from test_kernels_gpu import _ops, _rand

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _operands(dtype, T, W, n, seed):
    table = _rand((50, W), dtype, seed)
    values = [_rand((T, W), dtype, seed + 1 + k) for k in range(n)]
    ids = torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(seed)).int().cuda()
    ids[0] = 50                                 # outside: a row of zeros
    return ids, table, values


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,W,n", [(1, 4, 0), (3, 260, 1), (8, 2048, 6), (70, 4096, 15), (5, 1028, 9)])
def test_sources(dtype, T, W, n):
    ops = _ops()
    ids, table, values = _operands(dtype, T, W, n, 60 + n)
    weight = 1.0 + 0.1 * _rand((W,), torch.float32, 59)
    c = [0.7 - 0.3 * k for k in range(n + 1)]
    rows = torch.tensor([T - 1, 0], dtype=torch.int32, device=DEV)
    first = table.double()[ids.clamp(max=49).long()] * (ids < 50)[:, None]
    parts = [first] + [v.double() for v in values]
    c32 = torch.tensor(c, dtype=torch.float32).double().tolist()
    u = sum(w * p for w, p in zip(c32, parts))
    off = u - u.mean(dim=-1, keepdim=True)
    want = off * torch.rsqrt((off * off).mean(dim=-1, keepdim=True) + 1e-5) * weight.double()
    # n + 1 products and sums of numbers of the size of the largest part, then the norm: 2^-24 each of a row's spread; one rounding
    # to bfloat16 behind it
    size = sum(abs(w) * p.abs() for w, p in zip(c32, parts)) * torch.rsqrt((off * off).mean(dim=-1, keepdim=True) + 1e-5) * weight.double()
    bound = (2 * n + 16) * 2.0 ** -24 * size.amax(dim=-1, keepdim=True) + (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22) * want.abs()
    got = ops.read_sources(ids, table, values, c, weight, 1e-5)
    assert got.dtype == dtype and bool(((got.double() - want).abs() <= bound + 1e-30).all())
    assert torch.equal(ops.read_sources(ids, table, values, c, weight, 1e-5, rows=rows), got[rows.long()])
    each = _rand((3, n + 1), torch.float32, 58)
    x = ops.streams_from_sources(ids, table, values, each)
    for s in range(3):
        mine = [w * p for w, p in zip(each[s].double().tolist(), parts)]
        spread = sum(m.abs() for m in mine)
        assert bool(((x[:, s].double() - sum(mine)).abs() <= (n + 2) * 2.0 ** -24 * spread + 1e-30).all())


def test_what_is_refused():
    ops = _ops()
    ids, table, values = _operands(torch.bfloat16, 4, 256, 2, 40)
    weight = torch.ones(256, device=DEV)
    for bad in (lambda: ops.read_sources(ids, table, values, [1.0, 2.0], weight, 1e-5),
                lambda: ops.read_sources(ids, table, values * 8, [1.0] * 17, weight, 1e-5),
                lambda: ops.read_sources(ids, table, [values[0].float()], [1.0, 1.0], weight, 1e-5),
                lambda: ops.read_sources(ids, table[:, :254].contiguous(), [], [1.0], weight[:254], 1e-5)):
        with pytest.raises(ValueError):
            bad()


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("layers,streams", [(1, 2), (3, 4), (5, 4), (9, 3), (17, 4)])
def test_a_model_of_sources(dtype, layers, streams):
    from qwen3_from_scratch_amd.config.surasun_config import SurasunConfig
    from qwen3_from_scratch_amd.engine import ModelRunner, StepEntry, random_model
    from qwen3_from_scratch_amd.models.stream_sources import stream_plan

    width, dtype_asked = 128, dtype
    mamba = dict(heads=4, vdim=32, state=32, groups=1, conv=4, norm_groups=1)
    both = dict(left=dict(heads=2, kv_heads=2, dim=64, vdim=64, scale=0.125, softcap=50.0, rot=dict(dims=64, base=10000.0)),
                right=dict(heads=2, dim=32, vdim=64, rot=dict(dims=32, base=10000.0), decay=[0.9, 0.97]),
                left_scale=0.5, right_scale=0.75)
    config = SurasunConfig.from_dict({
        "architecture": "Surasun", "vocab": 300, "width": width, "norm": {"eps": 1e-5}, "residual_mult": 1.0, "streams": streams,
        "layers": [{"type": "parallel", "mixer": both, "mlp": {"kind": "dense", "ff": 256}} if i % 3 == 2 else
                   {"type": "mamba2", "mixer": mamba, "mlp": {"kind": "dense", "ff": 256} if i % 3 else None} for i in range(layers)]})
    steps = [[StepEntry("a", list(range(37)), [3, 36]), StepEntry("b", list(range(50, 55)), [])],
             [StepEntry("a", [7], [0]), StepEntry("b", [9], [0])], [StepEntry("b", [11, 12], [1])]]
    logits = []
    for sources, dtype in ((True, dtype), (False, dtype), (False, "float32")):
        model = random_model(config, dtype=dtype, device=DEV, seed=5, std=0.06)
        for layer in model.layers:               # streams that go on mostly as they are: random ones forget, and rounding grows
            for read, write, mix in layer.block.tables.values():
                mix.add_(torch.eye(streams, device=DEV))
        plan = model.stream_plan = stream_plan(model)
        assert plan is not None and (plan.streams is None) == (layers < 5 or (layers == 5 and dtype == "bfloat16"))
        if not sources:
            model.stream_plan = None
        runner = ModelRunner(model, 16, 32, max_requests=4)
        logits.append(torch.cat([runner.step(step).clone() for step in steps]))
    # the same weights in float32, to which either comes as near as the activations' dtype lets it
    got, streams, exact = logits
    bound = 1e-4 if dtype_asked == "float32" else 1.25 * float((streams - exact).norm() / exact.norm())
    assert float((got - exact).norm() / exact.norm()) <= bound
