"""Runs of layers that are alike.

The layers of a dense model differ in their weights and caches only: each asks the host for the same launches in the same order.
A layer asked for through Python costs the host some 15 us a launch, which is what bounds a short prompt of a small model; made
natively from another layer's (``ops.RepeatedLaunches``) it costs 40 in all. So of a run of such layers Python walks the first two and
the last, and the launches of the second, the first whose input norm the layer before prepared, are made again for those between.

A part whose launches follow from its sizes and its tensors alone says so: ``launch_key()``, equal for parts that launch alike
(None: not known), and ``launch_tensors()``, what they differ in, in an order of the part's own. Nothing is kept between steps: which runs
may be alike is known when the weights are, but a layer's key is asked for again in every step, since a part may have been given a
method, a number or a part of its own meanwhile (4 us a layer, while the GPU is at work on the one before).
"""
from __future__ import annotations

import functools

import torch

from ..kernels import ops

LEAST = 5  # layers of a run: with fewer there is none, or one, between those that Python walks

# Where the GPU takes longer for a layer than Python does, the GPU is what a step waits for, and looking at what may be made
# again, behind the second layer, leaves it idle for some 80 us. Estimated in us: weights from memory, multiply-adds, and what launches
# and attention take beside them. One prompt, every layer by Python / this way: 60 rows of the 0.6B shape 2,550 / 1,660 us, 487 rows 2,570 /
# 2,430 (the GPU's time), 90 of the 1.7B 2,610 / 2,340; slower so: 250 of the 4B 5,725 / 5,750, 40 of the 8B 4,205 / 4,285.
PYTHON_LAYER_US = 110.0
WEIGHT_BYTES_PER_US = 5.0e6
FLOPS_PER_US = {2: 0.8e9, 4: 1.0e8}  # by the weights' bytes an element
BESIDE_US = 25.0


def launches(x) -> bool:
    """Whether launches over the tensor are made now: on the GPU, and not into a graph."""
    return x.is_cuda and not torch.cuda.is_current_stream_capturing()


def key_of(part):
    """What the part says of its launches now (None: nothing)."""
    return part.launch_key() if hasattr(part, "launch_key") else None


def pays(layer, rows: int) -> bool:
    """Whether the host is what a step of so many rows waits for in such a layer."""
    if key_of(layer) is None:
        return False
    us = BESIDE_US
    for t in layer.launch_tensors():
        if t is not None and t.dim() == 2:
            us += t.nbytes / WEIGHT_BYTES_PER_US + 2.0 * rows * t.numel() / FLOPS_PER_US[t.element_size()]
    return us < PYTHON_LAYER_US


@functools.lru_cache(maxsize=None)
def _methods(kind):
    return frozenset(n for n in dir(kind) if not n.startswith("__") and callable(getattr(kind, n)))


def own_forward(part, kind) -> bool:
    """Whether the part is of exactly this class, with its methods."""
    return type(part) is kind and _methods(kind).isdisjoint(vars(part))


def equal_runs(schedule, layers):
    """For every run of the schedule the end of the stretch of runs, from it on, that launch alike."""
    keys = []
    for e in schedule:
        plain = e.cache_from is None and e.add_before is None and e.mix_before is None and not e.add_embedding
        keys.append(key_of(layers[e.layer]) if plain else None)
    ends = [0] * len(keys)
    for i in range(len(keys) - 1, -1, -1):
        same = i + 1 < len(keys) and keys[i] is not None and keys[i] == keys[i + 1]
        ends[i] = ends[i + 1] if same else i + 1
    return ends


def _tensors(layer, slot, next_norm):
    return [*layer.launch_tensors(), *(slot.rows[n] for n in sorted(slot.rows)), *next_norm.launch_tensors()]


def _form(t):
    """What the same launches need to be alike of a tensor that they are given: sizes, type, layout, place, the address's alignment."""
    return None if t is None else (t.shape, t.dtype, t.stride(), t.device, t.data_ptr() % 64)


def _carried(promise):
    return (promise.scaled, promise.partials, promise._rows) if type(promise) is ops.NormedRows else (None, None, None)


def walk(layers, slots, first, last, x, step, carry, next_norm_of):
    """Runs the layers ``first`` .. ``last`` - 1 (numbers of runs; ``layers`` and ``slots`` by run) as far as this pays and returns
    (the next run, its carry). ``next_norm_of(run)``: the norm that reads what the run leaves."""
    run = first
    carry = layers[run].forward(x, step, slots[run], normed_in=carry, next_norm=next_norm_of(run))
    run += 1
    norm, key = next_norm_of(run), key_of(layers[run])
    norm_key = key_of(norm)
    if key is None or norm_key is None:
        return run, carry
    own, taken = _tensors(layers[run], slots[run], norm), _carried(carry)
    with ops.kept_launches() as kept:
        left = layers[run].forward(x, step, slots[run], normed_in=carry, next_norm=norm)
    given, carry = _carried(left), left
    run += 1
    between = range(run, last - 1)
    if not kept.calls or type(left) is not ops.NormedRows or [_form(t) for t in taken] != [_form(t) for t in given]:
        return run, carry
    # what the kept launches took of the layer before and left for the next: the first of the others finds them the other way round
    turns = [(a, b) for a, b in zip(taken, given) if a is not None]
    here, there = [t.data_ptr() for pair in turns for t in pair], [t.data_ptr() for a, b in turns for t in (b, a)]
    spans = [(t.data_ptr(), t.data_ptr() + t.nbytes) if t is not None else (0, 0) for t in own] + [(a, a + 1) for a in here]
    again = ops.RepeatedLaunches(kept, spans)
    if not again.able:
        return run, carry
    forms, mine = [_form(t) for t in own], slots[run - 1]
    for n, run in enumerate(between):  # (one by one: the GPU is at work on one while the host looks at the next)
        slot, norm = slots[run], next_norm_of(run)
        if key_of(layers[run]) != key or key_of(norm) != norm_key:
            return run, carry
        tensors = _tensors(layers[run], slot, norm)
        if (slot.group, slot.writes, slot.page_size) != (mine.group, mine.writes, mine.page_size) or [_form(t) for t in tensors] != forms:
            return run, carry
        again.make([0 if t is None else t.data_ptr() for t in tensors] + (there if n % 2 == 0 else here))
        scaled, partials, normed = taken if n % 2 == 0 else given
        carry = ops.NormedRows(x, norm.gain, norm.eps, norm.out_dtype, scaled, partials)
        carry._rows = normed
    return last - 1, carry
