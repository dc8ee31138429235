"""How many blocks share a sequence's keys: always a number the kernels take, never more parts than there are
stretches of 64 keys, one part for short contexts; and at the sizes that its lines were drawn by, what was faster there,
for lengths as they are and for the powers of two that stand for them in captured steps."""

import pytest

from qwen3_from_scratch_amd import ops


@pytest.mark.parametrize("keys", [1, 64, 256, 257, 511, 512, 513, 1024, 2047, 2048, 4095, 4096, 8191, 8192, 65536, 1 << 20])
def test_splits_stay_in_range(keys):
    for requests in (1, 2, 4, 5, 16, 17, 24, 25, 32, 33, 40, 41, 48, 64, 65, 1000):
        for heads in (1, 2, 8, 40):
            splits = ops._splits(requests, heads, keys)
            assert 1 <= splits <= 64 and (splits == 1 or 64 * splits <= keys)
            assert splits == 1 or keys > 256


@pytest.mark.parametrize("requests,keys,parts", [
    (1, 256, 1), (1, 512, 8), (4, 512, 8), (8, 512, 1), (1, 1000, 15), (1, 8000, 32), (2, 4000, 16), (8, 2000, 4), (12, 2000, 2),
    (20, 1000, 1), (20, 1500, 1), (20, 2048, 1), (17, 2560, 3), (20, 2560, 3), (20, 4000, 3), (20, 4096, 3), (20, 6000, 3),
    (24, 2060, 1), (24, 4000, 1), (24, 4096, 1), (32, 6000, 1), (36, 1030, 1), (36, 1540, 3), (36, 2000, 3), (33, 2048, 3),
    (40, 6000, 3), (48, 2000, 1), (48, 4096, 1), (8, 7200, 8), (12, 8000, 8), (20, 8000, 8), (24, 8192, 8), (33, 8200, 8),
    (48, 7200, 4), (48, 32000, 4), (64, 8192, 1)])
def test_splits_that_were_faster(requests, keys, parts):
    assert ops._splits(requests, 8, keys) == parts


@pytest.mark.parametrize("rows,heads,kv_heads,dim,keys,pays", [
    (1, 16, 8, 128, 1100, True), (1, 16, 8, 128, 5000, True), (1, 32, 8, 128, 300, True), (2, 16, 8, 128, 450, True),
    (3, 8, 1, 128, 300, True), (2, 8, 1, 128, 1100, True), (2, 4, 4, 64, 3000, True), (4, 16, 8, 128, 300, False),
    (2, 32, 8, 128, 300, False), (1, 64, 8, 128, 300, False), (3, 4, 4, 64, 700, False), (6, 16, 16, 64, 700, False),
    (8, 8, 1, 128, 300, False), (16, 4, 4, 64, 1800, False), (1, 16, 8, 128, 200, False), (40, 16, 8, 128, 1000, False)])
def test_attention_that_is_best_merged_inside_the_product(rows, heads, kv_heads, dim, keys, pays):
    assert ops.split_rows_pay(rows, heads, kv_heads, dim, keys) == pays
