"""New requests' slots, neighbours or not, are zeroed on the GPU with as many operations as there are groups of states, and the host does not
wait for the device in between."""

from types import SimpleNamespace

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from qwen3_from_scratch_amd.cache.storage import CacheStorage

pytestmark = pytest.mark.gpu


class _Count(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.writes = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.writes += func._schema.name in ("aten::zero_", "aten::fill_", "aten::index_fill_", "aten::index_put_")
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("fresh", [[4], [3, 1, 2], [0, 7], list(range(0, 40, 2)), [39, 0, 1, 38]])
def test_slots(fresh):
    storage = CacheStorage.__new__(CacheStorage)
    storage.manager = SimpleNamespace(fresh_slots=list(fresh))
    storage.states = [torch.ones(2, 41, 3, device="cuda"), torch.ones(1, 41, 4, 2, device="cuda").bfloat16()]
    storage.device = torch.device("cuda:0")
    with _Count() as count:
        storage.clear_fresh_slots()
    assert count.writes == len(storage.states) and storage.manager.fresh_slots == []
    for t in storage.states:
        for slot in range(41):
            assert bool((t[:, slot] == (0 if slot in fresh else 1)).all())
