"""The last layer behind its mixer, for the rows that are wanted alone, against all rows."""
import pytest
import torch

import kebepel_tiny
import miforax_tiny
import tiny
from jllm_serve_amd.engine import StepEntry, build_runner, load_model
from jllm_serve_amd.kernels import ops
from jllm_serve_amd.parts import block
from jllm_serve_amd.parts.model import DecoderModel
from jllm_serve_amd.weights import write_random_model

pytestmark = pytest.mark.gpu

FAMILIES = {"qwen3": (tiny, "B"), "miforax": (miforax_tiny, "MA"), "miforax-experts": (miforax_tiny, "MB"), "kebepel": (kebepel_tiny, "KA"),
            "kebepel-wide": (kebepel_tiny, "KB")}


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("family", FAMILIES)
def test_logits_are_those_of_a_last_layer_over_all_rows(tmp_path, monkeypatch, family, dtype):
    """Steps that want no row, one, several of one request, and one of some of the requests beside single rows; each is followed by
    others that read the caches and states that the last layer wrote for all rows."""
    kind, name = FAMILIES[family]
    cfg, seed, page = kind.CONFIGS[name]
    folder = str(tmp_path / "model")
    (write_random_model if kind is tiny else kind.write_model)(folder, cfg, seed)
    steps = [[("a", 21, ())], [("a", 30, (29,)), ("b", 9, ())], [("c", 40, (0, 7, 39)), ("b", 5, (4,))], [("a", 1, (0,)), ("b", 25, ()), ("c", 1, (0,))],
             [("a", 1, (0,)), ("b", 1, (0,)), ("c", 1, ())], [("b", 12, (11, 3))]]
    monkeypatch.setattr(block, "WANTED_SAVE_US", {True: -1.0, False: -1.0})  # (these sizes save nothing)
    monkeypatch.setattr(block, "WANTED_LEAST_ROWS", {True: 0, False: 0})
    last = []
    for cls in {type(l) for l in load_model(folder, dtype, torch.device("cuda:0"), max_positions=256).layers}:
        if hasattr(cls, "forward_last"):
            monkeypatch.setattr(cls, "forward_last", lambda self, x, step, slot, normed_in=None, real=cls.forward_last:
                                last.append(step.n_selected) or real(self, x, step, slot, normed_in))

    def run(watch):
        model = load_model(folder, dtype, torch.device("cuda:0"), max_positions=256)
        model.watch = watch
        runner, gen, out = build_runner(model, page_size=page, pool_tokens=512, max_requests=4, graphs=False), torch.Generator().manual_seed(3), []
        for entries in steps:
            out.append(runner.step([StepEntry(rid, torch.randint(0, model.config.vocab, (n,), generator=gen).tolist(), want) for rid, n, want in entries]).clone())
        return out

    want = run(lambda run, x: None)  # a stream that is watched is whole in every layer
    assert not last
    got = run(None)
    assert last == [0, 1, 4, 2, 2, 2]
    for a, b in zip(got, want):
        assert a.shape == b.shape
        if a.numel():
            # both sides are within the family's bound of the plain implementation
            assert float((a.double() - b.double()).abs().max()) <= 2 * kind.tolerance(dtype, b.cpu().double())
    assert isinstance(load_model(folder, dtype, torch.device("cuda:0"), max_positions=256), DecoderModel)


@pytest.mark.parametrize("n", [1, 3, 200])
@pytest.mark.parametrize("width", [1, 7, 64, 2048, 2050])
def test_rows_are_gathered_as_they_are(n, width):
    """Row lengths of every unit that the kernel copies in, one, a few and many rows, with repeats and in any order, of contiguous matrices
    and of views that begin at an odd element, one to four at once."""
    gen = torch.Generator(device="cuda").manual_seed(n * width)
    held = [torch.randn(37, width + 3, device="cuda", generator=gen).to(t) for t in (torch.bfloat16, torch.float32, torch.bfloat16)]
    tensors = [held[0][:, 1:1 + width], held[1][:, :width], held[2][:, :width].contiguous(), torch.arange(37, device="cuda", dtype=torch.int32).view(-1, 1)]
    rows = torch.randint(0, 37, (n,), device="cuda", generator=gen, dtype=torch.int32)
    rows[0] = 36
    for k in (1, 2, 4):
        got = ops.gather_rows(rows, *tensors[:k])
        assert len(got) == k and all(torch.equal(g, t[rows.long()]) for g, t in zip(got, tensors))
    assert ops.gather_rows(rows[:0], *tensors)[1].shape == (0, width)
    with pytest.raises(ops.KernelError):
        ops.gather_rows(rows, *tensors, tensors[0])
