"""A Qwen3-shaped model over tensors that have sizes and no memory (device "meta"), with the launches of a step recorded in
place of being made: which kernel the host asks for, with which arguments, needs no GPU."""
import types

import torch

from jllm_serve_amd.config import parse_config
from jllm_serve_amd.engine.step import GroupStep, Segment, StepBatch, StepContext, StepPlan
from jllm_serve_amd.kernels import ops
from jllm_serve_amd.parts.model import DecoderModel


def tensor(*shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device="meta")


def record(monkeypatch):
    """From now on every launch is appended to the returned list as (entry point, arguments; tensors as themselves)."""
    seen = []
    monkeypatch.setattr(ops, "_try", lambda name, *args: seen.append((name, args)) or True)
    monkeypatch.setattr(ops, "_call", lambda name, *args: seen.append((name, args)))
    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_ptr", lambda t: t)
    return seen


def model(width, heads, kv_heads, ff, layers=2, dtype=torch.bfloat16):
    m = DecoderModel(parse_config({
        "architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_size": width, "num_hidden_layers": layers, "vocab_size": 4096,
        "num_attention_heads": heads, "num_key_value_heads": kv_heads, "head_dim": 128, "intermediate_size": ff, "rms_norm_eps": 1e-6,
        "rope_theta": 1e6, "tie_word_embeddings": False, "max_position_embeddings": 4096}), dtype, "meta", 4096)
    specs = {s.name: tuple(s.shape) for s in m.weight_specs()}
    m.load(types.SimpleNamespace(names=lambda: list(specs), shape=specs.get, get=lambda name: tensor(*specs[name], dtype=dtype)))
    return m


def forward(m, *requests, wanted=None):
    """One step of ``requests`` (rows, first position): its logits' rows are the requests' last ones, or ``wanted`` in number."""
    i32 = lambda *shape: tensor(*shape, dtype=torch.int32)
    segments, rows = [], 0
    for i, (n, pos0) in enumerate(requests):
        segments.append(Segment(i, i, rows, n, pos0, i))
        rows += n
    context = max(pos0 + n for n, pos0 in requests)
    batch = StepBatch(segments, rows, len(segments), context, 16, None, False)
    plans = {}
    for planner in m.step_planners():
        plan = planner.plan(batch)
        plans[planner.key] = StepPlan({name: i32(len(a)) for name, a in plan.arrays.items()}, plan.facts)
    wanted = len(segments) if wanted is None else wanted
    step = StepContext(rows, len(segments), i32(rows), i32(rows), i32(rows), i32(len(segments)), i32(wanted), wanted,
                       [GroupStep(i32(len(segments), -(-context // 16)), i32(rows))], segments, context, plans)
    slots = []
    for layer in m.layers:
        s = layer.mixer.spec
        pages = [tensor(64, s.kv_heads, 16, s.head_dim, dtype=m.dtype) for _ in range(2)]
        slots.append(types.SimpleNamespace(group=0, rows={"k": pages[0], "v": pages[1]}, writes=True, page_size=16))
    return m.forward(step, slots)
