"""Steps whose layers are launched natively against steps that Python walks layer by layer: the same bits."""
import types

import pytest
import torch

from jllm_serve_amd.config import parse_config
from jllm_serve_amd.engine import StepEntry, build_model, build_runner
from jllm_serve_amd.kernels import ops
from jllm_serve_amd.parts import equal_layers

pytestmark = pytest.mark.gpu


def runner_of(dtype, layers, width=512, ff=1024):
    config = parse_config({"architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_size": width, "num_hidden_layers": layers,
                           "vocab_size": 2048, "num_attention_heads": 4, "num_key_value_heads": 2, "head_dim": 128, "intermediate_size": ff,
                           "rms_norm_eps": 1e-6, "rope_theta": 1e6, "tie_word_embeddings": False, "max_position_embeddings": 2048})
    gen = torch.Generator(device="cuda").manual_seed(layers)
    from jllm_serve_amd.parts.model import DecoderModel
    shapes = {s.name: tuple(s.shape) for s in DecoderModel(config, torch.bfloat16, "meta", 2048).weight_specs()}
    stored = torch.float32 if dtype == "float32" else torch.bfloat16

    def get(name):
        t = torch.randn(shapes[name], device="cuda", generator=gen)
        return (1.0 + 0.1 * t if len(shapes[name]) == 1 else t * shapes[name][1] ** -0.5).to(stored)

    source = types.SimpleNamespace(names=lambda: list(shapes), shape=shapes.get, dtype=lambda name: stored, get=get)
    model = build_model(config, source, dtype, torch.device("cuda", 0), 2048)
    return build_runner(model, page_size=16, pool_tokens=4096, max_requests=8, graphs=False)


@pytest.mark.parametrize("dtype", ["bfloat16", "float32"])
@pytest.mark.parametrize("layers", [5, 6, 8])
def test_steps_have_the_bits_of_layers_walked_one_by_one(monkeypatch, dtype, layers):
    """Prompts alone and ragged, portions behind others, single rows beside them and alone (not captured): every logit, what is in the
    caches (the later steps read it), and the kernels that are counted as run."""
    monkeypatch.setattr(equal_layers, "PYTHON_LAYER_US", 1e9)
    steps = [[("a", 40)], [("b", 300), ("c", 7)], [("a", 1), ("b", 1)], [("a", 1), ("d", 130), ("c", 9)], [("d", 1)], [("e", 700)], [("a", 1), ("b", 1), ("c", 1), ("d", 1), ("e", 1)]]

    def run(least):
        monkeypatch.setattr(equal_layers, "LEAST", least)
        runner, gen, out = runner_of(dtype, layers), torch.Generator().manual_seed(1), []
        ops.reset_stats()
        for entries in steps:
            out.append(runner.step([StepEntry(rid, torch.randint(0, 2048, (n,), generator=gen).tolist(), (n - 1,)) for rid, n in entries]).clone())
        return out, ops.stats()["ran"]

    made = []
    make = ops.RepeatedLaunches.make
    monkeypatch.setattr(ops.RepeatedLaunches, "make", lambda self, addresses: (made.append(1), make(self, addresses)))
    want, ran = run(10 ** 6)
    assert not made
    got, ran_natively = run(5)
    assert len(made) == len(steps) * (layers - 3) and ran_natively == ran
    assert all(torch.equal(a, b) for a, b in zip(got, want)) and all(bool(torch.isfinite(a).all()) for a in got)


def test_a_layer_that_is_not_like_the_others_is_walked(monkeypatch):
    """Weights of another layout behind the same sizes, a part with a method of its own, and a function that watches the stream: no
    launch is taken from another layer where it might not be the same."""
    monkeypatch.setattr(equal_layers, "PYTHON_LAYER_US", 1e9)
    made = []
    make = ops.RepeatedLaunches.make
    monkeypatch.setattr(ops.RepeatedLaunches, "make", lambda self, addresses: (made.append(1), make(self, addresses)))
    runner, tokens = runner_of("bfloat16", 8), list(range(1, 31))

    def logits(rid):
        del made[:]
        got = runner.step([StepEntry(rid, tokens, range(30))]).clone()  # (every row: the last layer goes over all of them either way)
        runner.finish(rid)
        return got

    want = logits("a")
    assert len(made) == 5
    part = runner.model.layers[4].ffn
    held = torch.empty(part.w_down.numel() + 4, dtype=torch.bfloat16, device="cuda")
    kept, part.w_down = part.w_down, held[4:].view_as(part.w_down).copy_(part.w_down)  # 8 bytes behind a boundary of 16
    logits("b")
    assert len(made) == 2  # layers 2 and 3
    part.w_down = kept
    seen = []
    runner.model.watch = lambda run, x: seen.append(run)
    assert torch.equal(logits("c"), want) and seen == list(range(8)) and not made
    runner.model.watch = None
    part.forward = types.MethodType(type(part).forward, part)
    runner.model.equal_runs = equal_layers.equal_runs(runner.model.config.schedule, runner.model.layers)
    assert torch.equal(logits("d"), want) and not made
