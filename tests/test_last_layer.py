"""Where the last layer goes on with the wanted rows alone."""
import pytest
import torch

from jllm_serve_amd.config.schema import GatedMlpSpec, RoutedMoeSpec, TableMoeSpec
from jllm_serve_amd.parts.base import BuildContext, Part, part_factory
from jllm_serve_amd.parts.block import rows_alone

BUILD = BuildContext(64, torch.bfloat16, "cpu", 128)


class Neighbours(Part):
    """A feed-forward whose rows depend on other rows: it does not say ``rows_alone``."""

    def forward(self, xb, residual, step):
        residual += xb.float().roll(1, 0)


@pytest.mark.parametrize("spec", [TableMoeSpec(4, 2, 32, 7.0, 100, shared=GatedMlpSpec(hidden=32)), RoutedMoeSpec(4, 2, 32, shared=GatedMlpSpec(hidden=32))],
                         ids=lambda s: s.kind)
def test_a_shared_feed_forward_is_asked_too(spec):
    """Experts route every row by itself, but what runs beside them may be of any kind or have a method of its own."""
    ffn = part_factory("ffn", spec.kind)(spec, "l0", BUILD)
    assert rows_alone(ffn)
    ffn.shared.forward = lambda *args, **kw: None
    assert not rows_alone(ffn)
    del ffn.shared.forward
    assert rows_alone(ffn)
    ffn.shared = Neighbours()
    assert not rows_alone(ffn)
    ffn.shared = None
    assert rows_alone(ffn)
