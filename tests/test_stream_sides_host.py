"""A mixer between streams that are kept as the sums that they are: its results come apart if it can give them so, not because of what
it calls its own numbers."""

from types import SimpleNamespace

import pytest
import torch

from qwen3_from_scratch_amd.parts.base import Precision
from qwen3_from_scratch_amd.parts.block import HyperConnectionBlock


class _Mixer:
    def forward(self, h, batch, cache):
        return h + 1.0


class _Quantised(_Mixer):
    scales = torch.tensor([3.0, 5.0])      # of its own weights


class _Sides(_Mixer):
    scales = (0.5, 0.25)

    def forward_sides(self, h, batch, cache):
        return h + 1.0, h + 2.0


@pytest.mark.parametrize("mixer,scales", [(_Mixer(), (1.0,)), (_Quantised(), (1.0,)), (_Sides(), (0.5, 0.25))])
def test_whose_results_come_apart(mixer, scales):
    block = HyperConnectionBlock("b", Precision(torch.float32), torch.device("cpu"), 2)
    norm = SimpleNamespace(forward=lambda x, delta=None, read=None: torch.zeros(3, 4))
    block.attach(mixer=mixer, mixer_norm=norm)
    block.tables = {1: (torch.ones(2), torch.ones(2), torch.eye(2))}
    assert block.sublayer_scales() == [(1, scales)]
    _, apart = block.forward(SimpleNamespace(), None, None, None)
    assert tuple(apart.scales) == scales and isinstance(apart.values, tuple) == (len(scales) == 2)
    _, joined = block.forward(torch.zeros(3, 2, 4), None, None, None)
    assert torch.equal(joined.values, torch.ones(3, 4)) and joined.scales == (1.0,)
