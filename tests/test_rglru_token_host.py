"""The recurrent unit's step of one token a sequence: one kernel, but not where the kernels one by one were measured to be faster."""

import pytest

from qwen3_from_scratch_amd.ops.build import library


@pytest.mark.parametrize("rows,width,blocks,one", [
    (1, 2048, 8, True), (48, 2048, 8, True), (1, 512, 1, True), (16, 512, 1, True), (1, 1024, 2, True), (16, 4096, 8, True),
    (1, 640, 1, False), (1, 1024, 1, False), (32, 1024, 1, False), (33, 1024, 1, True), (16, 1152, 1, False), (17, 1152, 1, True),
    (16, 1536, 1, False), (17, 1536, 1, True), (1, 2560, 4, True), (1, 1536, 2, False), (17, 1536, 2, True), (1, 4096, 4, True),
    (1, 1552, 1, False), (0, 512, 1, False), (8, 512, 3, False)])
def test_the_faster_way(rows, width, blocks, one):
    assert bool(library("recurrent").q3_rglru_token_takes(rows, width, blocks)) == one
