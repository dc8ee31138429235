"""Products of 129 to 640 rows of a small weight that carry a norm, and the steps that are made of them."""

import pytest
import torch

from test_kernels_gpu import _forget_choices, _ops, _rand, rules_alone, test_linear_residual_norm_and_unscaled_rows_beyond_sixteen as _fused_products

pytestmark = pytest.mark.gpu


# rows at both ends of the range and of a tile; a writer that shares K out and one that does not; readers whose tiles fit
# the chip in one round of 64 x 128, of 128 x 128, and of neither
@pytest.mark.parametrize("M,H,K,N2", [(129, 1024, 2048, 4096), (256, 1024, 4096, 8192), (257, 1024, 4096, 8192),
                                      (400, 1088, 1024, 8000), (640, 1024, 4096, 8192), (640, 2048, 4096, 2560)])
@pytest.mark.parametrize("norm_dtype", [torch.float32, torch.bfloat16])
def test_products_that_carry_a_norm(M, H, K, N2, norm_dtype):
    _fused_products(M, H, K, N2, norm_dtype)


def test_rows_and_weights_that_take_part():
    ops = _ops()
    small, large, tiny = (torch.empty(n, 1024, dtype=torch.bfloat16, device="cuda") for n in (8192, 10240, 512))
    assert [ops.fused_rows_take(small, m) for m in (16, 17, 128, 129, 640, 641)] == [False, True, True, True, True, False]
    assert [ops.fused_rows_take(w, 129) for w in (large, tiny)] == [False, False]


def test_the_tuner_and_the_table_reach_640_rows(rules_alone):
    """Rows beyond 128 of small weights get entries of their own, those beyond 640 and those of a smaller weight do not; a
    size follows its entry, another keeps the rule."""
    from qwen3_from_scratch_amd.ops import tune

    ops = rules_alone
    ops.matmul_candidates(1)
    try:
        entries = tune.tune_layer(1088, 16, 8, 64, 2048, [256, 648])
    finally:
        ops.matmul_candidates(16)
    sizes = {kind: {(e["rows"], e["N"], e["K"]) for e in entries if e["kind"] == kind} for kind in ops._KINDS}
    assert sizes["scaled"] == {(256, 2048, 1088)} and sizes["scaled_swiglu"] == {(256, 4096, 1088)}
    assert sizes["residual"] == {(256, 1088, 1024), (256, 1088, 2048)}
    assert (648 + 31) // 32 * 32 in {rows for rows, _, _ in sizes["plain"]}

    M, N, K = 256, 2048, 1088
    x, w, sums = _rand((M, K), torch.bfloat16, 81), _rand((N, K), torch.bfloat16, 82, scale=0.05), torch.ones(2, M, device="cuda")
    want = (x.double() @ w.double().T) * (2.0 / K + 1e-6) ** -0.5
    _forget_choices(ops)
    beyond = ops.matmul_fused_plan("scaled", M + 8, N, K)
    for choice in ((1, 2), (0, 1), (-1, 1)):
        entry = {"kind": "scaled", "rows": ops.matmul_rows_key("scaled", M), "N": N, "K": K}
        entry.update(dict(library=0) if choice[0] < 0 else dict(own=choice[0], splits=choice[1]))
        ops.matmul_table([entry], clear=True)
        _forget_choices(ops)
        got = ops.linear(x, w, unscaled=(sums, 1e-6, K))
        assert ops.matmul_fused_plan("scaled", M, N, K) == choice
        torch.testing.assert_close(got.double(), want, rtol=1.6e-2, atol=1e-2)
        assert ops.matmul_fused_plan("scaled", M + 8, N, K) == beyond


def test_a_stream_too_wide_for_the_partial_products():
    """640 rows of 65,536 columns: the plain product and the norm's own kernel, whichever kernels are asked for."""
    ops = _ops()
    x, w = (torch.ones(n, 64, dtype=torch.bfloat16, device="cuda") for n in (640, 65536))
    residual = torch.zeros(640, 65536, device="cuda")
    for which in ("own", "both"):
        ops.matmul_kernels(which)
        try:
            assert ops.linear_residual_norm(x, w, None, residual, torch.ones(65536, device="cuda")) is None
        finally:
            ops.matmul_kernels("both")


@pytest.mark.parametrize("inner", [4096, 8192])       # 8,192: the gate and up product is too large, its neighbours are not
def test_prompts_whole_and_in_portions(inner, tmp_path):
    import plain_qwen3
    from helpers import off_by
    from qwen3_from_scratch_amd.config import ModelConfig
    from qwen3_from_scratch_amd.engine import StepEntry, load_runner
    from qwen3_from_scratch_amd.weights import write_random_model

    config = ModelConfig.from_dict(dict(
        architectures=["Qwen3ForCausalLM"], vocab_size=2048, hidden_size=1024, hidden_act="silu", num_hidden_layers=3,
        max_position_embeddings=2048, num_attention_heads=16, num_key_value_heads=8, head_dim=128,
        intermediate_size=inner, rms_norm_eps=1e-6, rope_theta=1e6, tie_word_embeddings=False))
    folder = write_random_model(str(tmp_path / "model"), config, seed=3)
    runner = load_runner(folder, dtype="bfloat16", device="cuda:0", page_size=16, max_tokens=1600, max_requests=2)
    tokens = torch.randint(0, 2048, (641,), generator=torch.Generator().manual_seed(4)).tolist()
    plain = plain_qwen3.logits_of_sequence(*plain_qwen3.read_model_folder(folder), tokens).cuda()

    def logits(cuts):
        at = 0
        for n in cuts:
            out = runner.step([StepEntry("r", tokens[at:at + n], [n - 1])])
            at += n
        out = out.clone()
        runner.finish("r")
        return out

    for M in (129, 300, 640, 641):
        whole = logits([M])
        portions = logits([100] * (M // 100) + [M % 100 or 100][:1] * bool(M % 100))
        # two bfloat16 ways through three layers: a few roundings of 2^-9 each
        assert float((whole - portions).norm() / portions.norm()) < 2e-2, M
        # and neither farther from a plain float32 pass than that
        for got in (whole, portions):
            assert off_by(got[0], plain[M - 1], "bfloat16") <= 1.0, M
            assert float((got[0] - plain[M - 1]).norm() / plain[M - 1].norm()) < 2e-2, M
