"""What a step asks the kernels for, from the shapes alone: launches recorded over tensors without memory."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

import recorded
from jllm_serve_amd.kernels import ops

SHAPES = {"0.6b": (1024, 16, 8, 3072), "1.7b": (2048, 16, 8, 6144), "4b": (2560, 32, 8, 9728)}  # width, heads, kv heads, feed-forward


@pytest.mark.parametrize("size", SHAPES)
def test_a_norm_is_prepared_only_where_its_reader_takes_it(monkeypatch, size):
    """The adding product of many rows leaves scaled rows and partial sums only for a product that reads them; and it is not
    credited for a norm that is a launch of its own."""
    seen = recorded.record(monkeypatch)
    m = recorded.model(*SHAPES[size], layers=3)
    rode = 0
    for rows in (17, 40, 64, 65, 127, 128, 200, 321, 400, 487, 512, 513, 600, 640, 750, 897, 960, 1009, 1024, 1500):
        del seen[:]
        recorded.forward(m, (rows, 0))
        left = read = 0
        for name, args in seen:
            if name == "jllm_gemm_stream_bf16":
                left += args[19] is not None   # emit_rows
                read += args[25] is not None   # norm_partial
            if name == "jllm_gemm_skinny_norm_bf16":  # the last layer's, of the wanted row
                left += args[15] is not None
                read += args[20] is not None
        assert left == read, (rows, left, read)
        rode += left
        norms = [args for name, args in seen if name == "jllm_rmsnorm"]
        made = sum(name in ("jllm_gemm_mfma_bf16", "jllm_gemm_pingpong_bf16") and args[-3] is not None for name, args in seen)
        assert len(norms) + made + left == 2 * 3 + 1, rows  # two norms a layer and the last one, each of them once
        rode -= 1  # (the wanted row's norm always rides)
    assert rode or size == "4b"


def test_no_norm_is_asked_for_when_its_reader_takes_rows_only():
    """A feed-forward that gathers its rows (routed experts) gets the norm as a launch: the product in front of it is not
    asked to prepare one that would be thrown away."""
    from types import SimpleNamespace
    from jllm_serve_amd.parts.block import PreNormBlock
    asked = []
    for takes in (False, True):
        block = PreNormBlock.__new__(PreNormBlock)
        block.ffn = SimpleNamespace(takes_normed_rows=takes, forward=lambda xb, x, step: None)
        block.mixer = SimpleNamespace(prepares_next_norm=True, forward=lambda xb, x, step, slot, then_norm=None: asked.append(then_norm))
        block.norm_in = SimpleNamespace(forward=lambda x: x)
        block.norm_post = SimpleNamespace(forward=lambda x: x, after_add=None, reader=block.ffn)
        block.forward("x", None, None)
    assert asked == [None, block.norm_post]


class Clears(TorchDispatchMode):
    """Counts the fill launches inside."""

    def __init__(self):
        super().__init__()
        self.n = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.n += func in (torch.ops.aten.zero_.default, torch.ops.aten.zeros.default, torch.ops.aten.fill_.Scalar)
        return func(*args, **(kwargs or {}))


def test_a_step_clears_counters_once_and_only_for_products_that_count(monkeypatch):
    """The products with K cut over workgroups share the step's counters, cleared for the first of them; a step that has none,
    in 32 bits or with every K whole, launches nothing for them."""
    with ops.step_scratch(40, torch.device("cuda")):
        pass  # nothing is made, so this needs no GPU
    seen = recorded.record(monkeypatch)
    for dtype, rows, counts in ((torch.bfloat16, 40, True), (torch.float32, 40, False), (torch.float32, 487, False), (torch.bfloat16, 16, False), (torch.bfloat16, 487, None)):
        m = recorded.model(*SHAPES["0.6b"], dtype=dtype)
        del seen[:]
        with Clears() as clears:
            recorded.forward(m, (rows, 0))
        counters = [args[18] for name, args in seen if name == "jllm_gemm_stream_bf16" and args[16] > 1]
        assert counts is None or bool(counters) == counts
        assert clears.n == bool(counters) and all(c is counters[0] for c in counters), (dtype, rows, clears.n)
