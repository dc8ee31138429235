"""Which steps Mamba-2's walk over the chunks' states takes: the ones that it was measured to be the faster way for."""

import pytest

from qwen3_from_scratch_amd.ops.build import library


@pytest.mark.parametrize("H,P,N,lengths,pays", [
    (64, 64, 128, [2048], True), (64, 64, 128, [8192], True), (64, 64, 128, [9], True), (16, 64, 128, [8192], True), (8, 64, 128, [4096], True),
    (8, 64, 128, [8192], False), (1, 64, 128, [2048], True), (1, 64, 128, [4096], False), (4, 64, 128, [16384], False),
    (8, 64, 64, [1024], True), (8, 64, 64, [2048], False), (24, 64, 64, [8192], True), (16, 64, 64, [8192], False),
    (8, 64, 256, [4096], True), (4, 64, 256, [8192], False), (48, 64, 32, [8192], True), (24, 64, 32, [8192], False), (1, 16, 32, [1024], False),
    (4, 32, 32, [256], True), (4, 32, 32, [8192], False), (4, 32, 32, [2048] + [1] * 16, True), (64, 64, 128, [512] + [1] * 40, True)])
def test_steps_that_are_faster_so(H, P, N, lengths, pays):
    lib = library("mamba2")
    assert lib.q3_mamba2_walk_takes(H, P, N, 1)
    assert bool(lib.q3_mamba2_walk_pays(sum(lengths), len(lengths), max(lengths), H, P, N)) == pays


def test_any_size_has_an_answer():
    lib = library("mamba2")
    for T, B, longest in ((1, 1, 1), (1 << 30, 65535, 1 << 30), (64, 64, 1), (1 << 20, 1, 1 << 20)):
        for H, P, N in ((1, 16, 32), (1 << 12, 1 << 12, 256)):
            assert lib.q3_mamba2_walk_pays(T, B, longest, H, P, N) in (0, 1)
