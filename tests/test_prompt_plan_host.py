"""How a step's prompts go over blocks (a host function of the attention library): at the sizes that its lines were drawn by what was
faster there, whatever else is in the step, and for a group of more heads than the kernels take an answer too."""

import pytest

from qwen3_from_scratch_amd.ops.build import library


def _plan(heads, lengths, keys, window=0):
    """Rows of a block, whether a mixed launch has the prompts first, whether sixteen rows a block serve; parts of the keys."""
    from qwen3_from_scratch_amd import ops

    H, G = heads
    T, B, longest = sum(lengths), len(lengths), max(k for n, k in zip(lengths, keys) if n > 1)
    splits = ops._splits(B, G, max(keys)) if min(lengths) * (H // G) <= 16 else 1
    lib = library("attention")
    parts = lib.q3_paged_attention_prompt_splits(T, H, G, longest)
    plan = lib.q3_paged_attention_plan(T, B, H, G, parts, splits, window, max(lengths), min(lengths), longest, max(keys))
    return plan % 256 * (H // G), bool(plan & 256), bool(plan & 512), parts


def _spread(n, low, high):
    return [high - (high - low) * i // max(1, n - 1) for i in range(n)]


@pytest.mark.parametrize("heads,lengths,keys,rows,parts", [
    # what is left over at each prompt's end counts
    ((32, 8), [70] * 16, [70] * 16, 128, 1), ((16, 8), [130] * 16, [130] * 16, 128, 1), ((32, 8), [130] * 8, [130] * 8, 128, 1),
    ((64, 8), [128] * 4, [128] * 4, 128, 1), ((16, 8), [300] * 7, [300] * 7, 128, 1), ((16, 8), [270] * 8, [270] * 8, 128, 1),
    # long chains, few rows
    ((32, 8), [1100], [1100], 64, 1), ((16, 8), [2300], [2300], 64, 1), ((32, 8), [512], [512], 32, 1), ((32, 8), [64] * 8, [64] * 8, 32, 1),
    ((8, 8), [20] * 64, [20] * 64, 32, 1), ((32, 8), [2048], [2048], 128, 1), ((32, 8), [8192], [8192], 128, 1), ((32, 8), [1024], [1024], 64, 1),
    # parts of the keys
    ((16, 8), [276], [2300], 32, 2), ((32, 8), [276], [3100], 32, 1), ((32, 8), [128], [2048], 32, 1), ((32, 8), [512], [8000], 128, 4)])
def test_prompts(heads, lengths, keys, rows, parts):
    found = _plan(heads, lengths, keys)
    assert (found[0], found[3]) == (rows, parts)


@pytest.mark.parametrize("heads,singles,portions,rows,first", [
    ((32, 8), _spread(40, 150, 3000), [(512, 512)], 128, False), ((16, 8), _spread(40, 150, 3000), [(512, 512)], 64, False),
    ((32, 8), _spread(48, 150, 3000), [(512, 512)], 128, False), ((32, 8), _spread(32, 150, 3000), [(512, 1536)], 64, True),
    ((32, 8), _spread(23, 150, 3000), [(276, 1300)], 64, True), ((32, 8), _spread(28, 150, 3000), [(1400, 1400)], 128, True),
    ((16, 8), _spread(28, 150, 3000), [(300, 300)] * 4, 128, False), ((32, 8), _spread(23, 150, 3000), [(512, 3584)], None, None),
    ((64, 8), _spread(40, 150, 3000), [(1400, 1400)], 128, False), ((64, 8), _spread(64, 200, 1000), [(1400, 1400)], 128, True),
    ((16, 8), _spread(30, 150, 500), [(16, 16), (33, 33), (51, 51)], 32, True),
    # one decoding request among prompts is not as many as there are sequences
    ((32, 8), [3000], [(130, 130)] * 15, 128, False), ((32, 8), [150], [(33, 33)] * 30, 128, True), ((16, 8), [150], [(300, 300)] * 7, 128, True)])
def test_prompts_beside_decoding_requests(heads, singles, portions, rows, first):
    found = _plan(heads, [1] * len(singles) + [n for n, _ in portions], singles + [k for _, k in portions])
    if rows is None:             # parts of the keys that fill the chip by themselves
        assert found[3] == 1 or not found[1]
    else:
        assert found[:3] == (rows, first, False)


@pytest.mark.parametrize("heads,lengths,keys,brief", [
    ((16, 8), [200], [200], True), ((32, 8), [200], [200], False), ((16, 8), [300], [300], False), ((32, 8), [32], [1900], True),
    ((32, 8), [1] * 36 + [20], [150] * 36 + [820], True), ((32, 8), [1] * 16 + [100], [150] * 16 + [900], True),
    ((32, 8), [1] * 28 + [20], _spread(28, 150, 3000) + [820], False), ((8, 8), [500, 20, 20, 20], [500, 20, 20, 20], True),
    ((8, 8), [300, 300], [300, 300], False)])
def test_few_rows(heads, lengths, keys, brief):
    assert _plan(heads, lengths, keys)[2] == brief


@pytest.mark.parametrize("build", ["attention", "attention_capped", "attention_capped_gated", "attention_pooled", "attention_sigmoid", "attention_span"])
@pytest.mark.parametrize("group", [1, 16, 33, 64, 129, 500])
def test_any_group_of_heads_has_an_answer(build, group):
    lib = library(build)
    for keys in (100, 2048, 2600, 5000, 100000):
        assert lib.q3_paged_attention_prompt_splits(700, 2 * group, 2, keys) in (1, 2, 4)
    assert lib.q3_paged_attention_plan(700, 3, 34, 2, 1, 1, 0, 300, 1, 300, 300) == 0      # 17 heads a group: not the fast path's


def test_capped_scores_without_a_gate_carry_none():
    assert not hasattr(library("attention_capped"), "q3_set_gate") and hasattr(library("attention_capped_gated"), "q3_set_gate")
