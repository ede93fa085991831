"""Where the last layer goes on with the wanted rows alone."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import recorded
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


class Noted(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, kinds, args=(), kwargs=None):
        self.names.append(func.overloadpacket.__name__)
        return func(*args, **(kwargs or {}))


@pytest.mark.parametrize("rows", [40, 300])
def test_the_wanted_rows_are_taken_by_one_launch(monkeypatch, rows):
    """The heads' rows and the stream's together, by the project's own kernel; token ids are not gathered for a feed-forward that
    does not read them; and the norm behind the o product is made on its way, as in every other layer."""
    m = recorded.model(4096, 32, 8, 12288, layers=2)
    seen = recorded.record(monkeypatch)
    with Noted() as noted:
        recorded.forward(m, (rows, 0), (1, 9))
    names = [name for name, _ in seen]
    assert names.count("jllm_gather_rows") == 1 and names.count("jllm_embed") == 1
    assert names[-1].startswith("jllm_gemm") and names.count("jllm_rmsnorm") == 2  # in front of the layers and behind them
    assert not {"index_select", "index", "gather", "take"} & set(noted.names), noted.names
    _, n_matrices, picked, n, height, _ = next(args for name, args in seen if name == "jllm_gather_rows")
    assert (n_matrices, n, height) == (2, 2, rows + 1)


def test_a_portion_that_wants_nothing_ends_with_the_cache(monkeypatch):
    """Of the last layer only what its cache gets is made; for single rows that is inside their attention's launch."""
    m = recorded.model(4096, 32, 8, 12288, layers=2)
    seen = recorded.record(monkeypatch)
    for requests, last in (([(300, 0), (1, 9)], "jllm_qk_norm_rope_store"), ([(1, 9), (1, 30)], "jllm_decode_attention_fused_bf16")):
        del seen[:]
        assert recorded.forward(m, *requests, wanted=0).shape == (0, 4096)
        names = [name for name, _ in seen]
        assert names[-1] == last and names.count(last) == 2, names


def test_rows_are_taken_apart_only_where_that_saves_something(monkeypatch):
    """Steps that drop few rows, and those of few rows altogether, keep the last layer whole: no gather, and the final norm takes the
    row list; a prompt whose last row is wanted does not."""
    m = recorded.model(1024, 16, 8, 3072, layers=2)
    seen = recorded.record(monkeypatch)

    def apart(*requests, wanted=None):
        del seen[:]
        recorded.forward(m, *requests, wanted=wanted)
        picked = [args for name, args in seen if name == "jllm_rmsnorm"][-1][1]
        some = any(name == "jllm_gather_rows" for name, _ in seen)
        assert some == (picked is None)
        return some

    assert not any(apart((n, 0)) for n in (2, 5, 16))
    assert not apart(*[(1, 100)] * 64, wanted=63) and not apart((100, 0), wanted=99) and not apart(*[(1, 9)] * 2, wanted=1)
    assert all(apart((n, 0)) for n in (17, 64, 300, 2000)) and apart((300, 0), (1, 9))
