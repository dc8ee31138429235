"""The slots of new requests are zeroed, and only they, whatever their order and neighbours."""

from types import SimpleNamespace

import pytest
import torch

from qwen3_from_scratch_amd.cache.storage import CacheStorage


@pytest.mark.parametrize("fresh", [[], [0], [5], [3, 1, 2], [0, 2, 4, 5], [1, 1, 0]])
def test_slots(fresh):
    storage = CacheStorage.__new__(CacheStorage)
    storage.manager = SimpleNamespace(fresh_slots=list(fresh))
    storage.states = [torch.ones(2, 6, 3), torch.ones(1, 6, 4, 2)]
    storage.clear_fresh_slots()
    assert storage.manager.fresh_slots == []
    for t in storage.states:
        for slot in range(6):
            assert bool((t[:, slot] == (0 if slot in fresh else 1)).all())
