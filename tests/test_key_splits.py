"""How many blocks share a sequence's keys: always a number the kernels take, never more parts than there are
stretches of 64 keys, one part for short contexts."""

import pytest

from qwen3_from_scratch_amd import ops


@pytest.mark.parametrize("keys", [1, 64, 256, 257, 511, 512, 513, 1024, 2047, 2048, 4095, 4096, 8191, 8192, 65536, 1 << 20])
def test_splits_stay_in_range(keys):
    for requests in (1, 2, 4, 5, 16, 17, 24, 25, 32, 33, 40, 41, 48, 64, 65, 1000):
        for heads in (1, 2, 8, 40):
            splits = ops._splits(requests, heads, keys)
            assert 1 <= splits <= 64 and (splits == 1 or 64 * splits <= keys)
            assert splits == 1 or keys > 256
