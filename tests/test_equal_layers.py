"""Layers whose launches are made natively from another layer's: the same launches, over the same data."""
import copy
import ctypes
import os
import re
import struct
import types

import pytest
import torch

import recorded
from jllm_serve_amd.kernels import build, ops
from jllm_serve_amd.parts import equal_layers
from jllm_serve_amd.parts.model import DecoderModel

WRITTEN = {"out", "emit_rows", "emit_partial", "partial", "norm_rows", "part_acc", "part_ml", "qkv", "kcache", "vcache"}


def parameters():
    """Entry point -> names of its parameters, as the sources have them."""
    with open(os.path.join(build.SRC_DIR, "layer_launches.h")) as f:
        text = re.sub(r"\s+", " ", f.read())
    return {name: [a.split()[-1].lstrip("*") for a in args.split(",")] for name, args in re.findall(r"int (\w+)\(([^)]*)\);", text)}


class Library:
    """Stands in for the kernel library: calls are noted, with addresses as numbers, and nothing runs."""

    def __init__(self):
        self.names, self.calls = sorted(parameters()), []

    def jllm_layer_entry(self, name, count):
        return self.names.index(name.decode()) if count == len(parameters()[name.decode()]) else -1

    def jllm_layer_launches(self, words, n, places, n_places, values):
        for p in range(n_places):
            words[places[p]] = values[p]
        at = 0
        while at < n:
            name, count = self.names[words[at]], words[at + 1]
            types = ops._SIGS.get(name) or ops._OPTIONAL_SIGS[name]
            args = []
            for w, t in zip(words[at + 2:at + 2 + count], types):
                if t is ctypes.c_float:
                    args.append(struct.unpack("<f", struct.pack("<I", w))[0])
                else:
                    args.append(w if t is ctypes.c_void_p else ctypes.c_int(w & 0xFFFFFFFF).value)
            self.calls.append((name, tuple(args), True))
            at += 2 + count
        return 0

    def __getattr__(self, name):
        def entry(*args):
            self.calls.append((name, tuple(a if a is not None else 0 for a in args), False))
            return 0
        return entry


def data_flow(calls, tensors):
    """Every call with its addresses told by what lies there: a tensor of the model, what an earlier call wrote there, or (the
    step's arrays and tables) the place itself."""
    spans = sorted((t.data_ptr(), t.data_ptr() + t.nbytes, name) for name, t in tensors.items())
    wrote, seen, names = {}, [], parameters()
    for number, (name, args, _) in enumerate(calls):
        types = ops._SIGS.get(name) or ops._OPTIONAL_SIGS[name]
        told = []
        for what, a, t in zip(names.get(name, [""] * len(args)), args, types):
            if t is not ctypes.c_void_p or not a:
                told.append(ctypes.c_float(a).value if isinstance(a, float) else a)
                continue
            inside = [(n, a - begin) for begin, end, n in spans if begin <= a < end]
            told.append(inside[0] if inside else ("written by", *wrote[a]) if a in wrote else ("new",) if what in WRITTEN else ("at", a))
        for place, (what, a, t) in enumerate(zip(names.get(name, []), args, types)):
            if what in WRITTEN and t is ctypes.c_void_p and a:
                wrote[a] = (number, place)
        # (memory that a call only writes may be new or what an earlier layer wrote: not part of what it reads)
        plain = {"out", "emit_rows", "emit_partial", "partial", "norm_rows", "part_acc", "part_ml"}
        adds = "epilogue" in names.get(name, []) and args[names[name].index("epilogue")] == ops.EPI_ADD
        seen.append((name, tuple("written" if w in plain and not (w == "out" and adds) and isinstance(x, tuple) and x[0] in ("new", "written by") else x
                                 for w, x in zip(names.get(name, [""] * len(told)), told))))
    return seen


def stand_ins(monkeypatch, layers, dtype):
    """A model on the CPU whose launches are noted (every layer of it natively where it may be), its library, and all that was
    given to a launch (kept, so that no memory is given out twice and an address says which tensor)."""
    held = []
    monkeypatch.setattr(recorded, "tensor", lambda *shape, dtype=torch.bfloat16: held.append(torch.zeros(shape, dtype=dtype)) or held[-1])
    monkeypatch.setattr(recorded, "DecoderModel", lambda config, dtype, device, positions: DecoderModel(config, dtype, "cpu", positions))
    m = recorded.model(1024, 4, 2, 512, layers=layers, dtype=dtype)
    library = Library()
    monkeypatch.setattr(ops, "library", lambda: library)
    monkeypatch.setattr(ops, "_dev", lambda *tensors: None)
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(ops, "_layer_entries", {})
    monkeypatch.setattr(equal_layers, "launches", lambda x: True)
    monkeypatch.setattr(equal_layers, "PYTHON_LAYER_US", 1e9)
    real = ops._ptr
    monkeypatch.setattr(ops, "_ptr", lambda t: held.append(t) or real(t))
    return m, library, held


@pytest.mark.parametrize("layers", [5, 6, 9, 10])
@pytest.mark.parametrize("dtype,requests", [(torch.bfloat16, [(40, 0)]), (torch.bfloat16, [(487, 0)]), (torch.bfloat16, [(1, 9), (1, 30)]),
                                            (torch.bfloat16, [(300, 0), (1, 20), (1, 7)]), (torch.float32, [(3, 0)]), (torch.float32, [(100, 0)])])
def test_the_launches_and_what_they_read_are_those_of_every_layer_by_itself(monkeypatch, layers, dtype, requests):
    """For prompts, single rows and both, one layer beyond the least up to several, an even and an odd number of layers between: the
    same entry points with the same numbers, every address in the same tensor of the same layer or where the same earlier call wrote."""
    m, library, held = stand_ins(monkeypatch, layers, dtype)
    tensors = {(i, n): t for i, layer in enumerate(m.layers) for n, t in enumerate(layer.launch_tensors()) if t is not None}

    caches, forward = {}, type(m).forward

    def noting_caches(self, step, slots):
        caches.update({("cache", i, n): t for i, s in enumerate(slots) for n, t in s.rows.items()})
        return forward(self, step, slots)

    monkeypatch.setattr(type(m), "forward", noting_caches)

    def told(least):
        monkeypatch.setattr(equal_layers, "LEAST", least)
        library.calls.clear()
        caches.clear()
        recorded.forward(m, *requests)
        return data_flow(library.calls, {**tensors, **caches}), sum(native for _, _, native in library.calls)

    one_by_one, none = told(10 ** 6)
    native, some = told(5)
    assert none == 0 and some % (layers - 3) == 0 and some > 0
    at = lambda calls: [(n, tuple("step" if isinstance(x, tuple) and x[0] == "at" else x for x in args)) for n, args in calls]
    assert at(native) == at(one_by_one)


def with_a_limit(part):
    part.limit = 3.0


def with_a_method(part):
    part.forward = types.MethodType(type(part).forward, part)


CHANGES = {"a method of the feed-forward": lambda layer: with_a_method(layer.ffn), "a method of the layer": with_a_method,
           "a method of the norm": lambda layer: setattr(layer.norm_in, "after_add", types.MethodType(type(layer.norm_in).after_add, layer.norm_in)),
           "the norm's number": lambda layer: setattr(layer.norm_post, "eps", 1e-3), "the gate's limit": lambda layer: with_a_limit(layer.ffn),
           "another feed-forward": lambda layer: setattr(layer, "ffn", copy.copy(layer.ffn)) or with_a_limit(layer.ffn)}


@pytest.mark.parametrize("change", CHANGES)
@pytest.mark.parametrize("at", [1, 4])
def test_a_layer_that_was_changed_after_the_load_is_walked(monkeypatch, change, at):
    """What a program does to one layer of a loaded model is asked for by its own walk, whether that layer is the one whose launches
    would be kept or one of those between."""
    m, library, _ = stand_ins(monkeypatch, 9, torch.bfloat16)
    walked = []
    # (a layer that Python walks asks for the step's facts)
    real = type(m.layers[0].mixer)._batch_facts
    monkeypatch.setattr(type(m.layers[0].mixer), "_batch_facts", lambda self, *a: walked.append([l.mixer for l in m.layers].index(self)) or real(self, *a))
    recorded.forward(m, (40, 0))
    assert walked == [0, 1, 8]
    plain = library.calls[:]
    CHANGES[change](m.layers[at])
    walked.clear()
    library.calls.clear()
    recorded.forward(m, (40, 0))
    # (the norm of a changed layer is made by the layer before it)
    assert at in walked and (at == 4 or 2 in walked) and ("norm" not in change or "number" in change or at - 1 in walked)
    assert [c[0] for c in library.calls] == [c[0] for c in plain]
