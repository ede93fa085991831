"""Miforax on the GPU against the plain implementation (tests/plain/miforax_plain.py): every mechanism alone, the
attention kernels on crafted keys (far keys, window edges, page borders, sinks), whole prompts against token-by-token
decoding, portions down to two tokens, mixed batches on a pool that is used again, long decoding through captured
steps, greedy generation through the engine, and the replay program."""
import json
import os
import random

import numpy as np
import pytest
import torch

import miforax_tiny as mt
import replay
from plain import miforax_plain as P

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def built(miforax_folders):
    from jllm_serve_amd.engine import build_runner, load_model
    cache = {}

    def get(name, dtype):
        if (name, dtype) not in cache:
            model = load_model(miforax_folders[name], dtype, torch.device(DEV), max_positions=1024)
            cache[(name, dtype)] = (model, build_runner(model, page_size=mt.CONFIGS[name][2], pool_tokens=1024,
                                                        max_requests=4, graphs=False))
        return cache[(name, dtype)]
    return get


@pytest.fixture(scope="module")
def plain_logits(miforax_folders):
    memo = {}

    def get(name, tokens):
        key = (name, tuple(tokens))
        if key not in memo:
            memo[key] = P.forward(mt.CONFIGS[name][0], mt.load_weights(miforax_folders[name]), list(tokens))
        return memo[key]
    return get


def close(got, want, dtype, what=""):
    err = float((got.double().cpu() - want).abs().max())
    assert err <= mt.tolerance(dtype, want), f"{what}: {err} > {mt.tolerance(dtype, want)}"


# ------------------------------------------------------------------------------------------------ mechanisms alone


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["MA", "MB", "MC"])
def test_feed_forwards_alone(name, dtype, built, miforax_folders):
    from jllm_serve_amd.engine.step import StepEntry
    cfg = mt.CONFIGS[name][0]
    w = mt.load_weights(miforax_folders[name])
    model, runner = built(name, dtype)
    act = torch.float32 if dtype == "float32" else torch.bfloat16
    torch.manual_seed(3)
    for T in (1, 7, 45, 600):  # 600 rows give MB's experts enough rows each for the tiles of many rows
        toks = mt.prompt(name, T, seed=T)
        ctx = runner.prepare([StepEntry("ff", toks, [])])
        xb = (torch.randn(T, cfg["width"]) * 1.5).to(act)  # large enough that the experts' clamps bite
        res = torch.randn(T, cfg["width"])
        for i, layer in enumerate(cfg["layers"]):
            mlp = layer["mlp"]
            if mlp is None:
                assert model.layers[i].ffn is None
                continue
            r = res.clone().to(DEV)
            model.layers[i].ffn.forward(xb.to(DEV), r, ctx)
            if mlp["kind"] == "dense":
                want = res.double() + P.dense_ff(xb.double(), w, f"l{i}.mlp.")
            else:
                want = res.double() + P.table_moe(xb.double(), toks, w, f"l{i}.mlp.", mlp)
            close(r, want, dtype, f"{name} layer {i} feed-forward, {T} rows")
        runner.finish("ff")


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["MA", "MB", "MC"])
def test_mixers_alone_through_the_cache(name, dtype, built, miforax_folders):
    """Every layer's mixer on random inputs: a portion from position 0, a second portion and single rows from the
    cache; a layer that borrows a cache reads what its owner stored from the owner's own input."""
    from jllm_serve_amd.engine.step import StepEntry
    cfg = mt.CONFIGS[name][0]
    eps = cfg["norm"]["eps"]
    w = mt.load_weights(miforax_folders[name])
    model, runner = built(name, dtype)
    act = torch.float32 if dtype == "float32" else torch.bfloat16
    torch.manual_seed(4)
    cuts = (29, 6, 1, 1, 17)
    T = sum(cuts)
    xs = [(torch.randn(T, cfg["width"]) * 0.8).to(act) for _ in cfg["layers"]]
    pos = torch.arange(T)
    kept, want = {}, []
    for i, layer in enumerate(cfg["layers"]):
        m, p = layer["mixer"], f"l{i}.mix."
        if m.get("kv_from") is None:
            kept[i] = P.latent_kv(xs[i].double(), w, p, m, eps, pos)
        c, kr = kept[i if m.get("kv_from") is None else m["kv_from"]]
        want.append(P.latent_attention(xs[i].double(), w, p, m, eps, pos, c, kr))
    got = [[] for _ in cfg["layers"]]
    at = 0
    for n in cuts:
        ctx = runner.prepare([StepEntry("mix", [0] * n, [])])
        for i in range(len(cfg["layers"])):
            res = torch.zeros(n, cfg["width"], device=DEV)
            model.layers[i].mixer.forward(xs[i][at:at + n].to(DEV), res, ctx, runner.cache.slots[i])
            got[i].append(res.cpu())
        runner.cache.commit("mix", n)
        at += n
    runner.finish("mix")
    for i in range(len(cfg["layers"])):
        close(torch.cat(got[i]), want[i], dtype, f"{name} layer {i} mixer")


@pytest.mark.parametrize("gate, limit", [("silu", 0.0), ("gelu_tanh", 0.0), ("swish_clamped", 0.6), ("swish_clamped", 7.0)])
def test_gate_functions_in_every_product_kernel(gate, limit):
    """The gated product with each gate function at row counts that take each product kernel, in both types."""
    from jllm_serve_amd.kernels import ops
    torch.manual_seed(5)

    def ref(g, u):
        if gate == "silu":
            return g * torch.sigmoid(g) * u
        if gate == "gelu_tanh":
            return P.gelu_tanh(g) * u
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(1.702 * g) * (u + 1)

    for M, N, K in ((3, 256, 256), (40, 256, 256), (200, 384, 128), (600, 2048, 128), (5, 72, 40)):
        a = torch.randn(M, K).to(torch.bfloat16)
        wg, wu = (torch.randn(N, K) * 0.15).to(torch.bfloat16), (torch.randn(N, K) * 0.15).to(torch.bfloat16)
        want = ref(a.double() @ wg.double().T, a.double() @ wu.double().T)
        for dtype in ("float32", "bfloat16"):
            t = torch.float32 if dtype == "float32" else torch.bfloat16
            out = ops.gemm(a.to(DEV).to(t), wg.to(DEV).to(t), w2=wu.to(DEV).to(t), epilogue=ops.EPI_GATED, out_dtype=t,
                           exact=dtype == "float32", gate=ops.GATE_FUNCTIONS[gate], gate_limit=limit)
            close(out, want, dtype, f"{gate} {M}x{N}x{K}")


# ------------------------------------------------------------------------------------------------ crafted keys


def _attend_plain(qa, rows, R, window, scale, sink, q_pos):
    """float64: qa [T, H, Dk], rows [L, Dk] (position = index), q_pos [T]; returns [T, H, R]."""
    s = torch.einsum("thd,jd->thj", qa, rows) * scale
    j = torch.arange(rows.shape[0])[None, :]
    seen = (j <= q_pos[:, None]) & ((q_pos[:, None] - j < window) if window else torch.ones_like(j, dtype=torch.bool))
    s = s.masked_fill(~seen[:, None, :], float("-inf"))
    e = torch.exp(s - s.amax(-1, keepdim=True))
    den = e.sum(-1, keepdim=True) + (torch.exp(sink[None, :, None] - s.amax(-1, keepdim=True)) if sink is not None else 0)
    return torch.einsum("thj,jr->thr", e / den, rows[:, :R])


@pytest.mark.parametrize("N,K,tail,gated", [(512, 128, 64, False), (128, 512, 0, True), (36, 64, 24, False), (132, 192, 0, True),
                                            (20, 40, 8, False), (100, 256, 0, True), (68, 320, 16, False)])
def test_heads_products_at_every_row_count(N, K, tail, gated):
    """The per-head products where their kernel changes (up to 16 rows, up to 40 with a tail, tiles of 64 or 128 rows beyond) and at odd
    sizes: against float64, and a row's bits are those it has in any other batch."""
    from jllm_serve_amd.kernels import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    H, M = 3, 261
    x = torch.randn(M, H * (K + tail), device="cuda", generator=gen).bfloat16()
    w = (torch.randn(H, N, K, device="cuda", generator=gen) * K ** -0.5).bfloat16()
    gate = torch.randn(M, H * N, device="cuda", generator=gen).bfloat16() if gated else None
    positions = torch.arange(5, 5 + M, dtype=torch.int32, device="cuda")
    rot = tail // 8 * 8
    angle = torch.rand(M + 5, rot // 2, device="cuda", generator=gen) * 6.0
    cos, sin = torch.cos(angle), torch.sin(angle)

    def heads(n):
        return ops.latent_heads(x[:n].contiguous(), w, tail=tail, rot_dims=rot, positions=positions[:n].contiguous(),
                                cos=cos if tail else None, sin=sin if tail else None, gate=gate[:n].contiguous() if gated else None)

    whole = heads(M)
    for n in (1, 16, 17, 40, 41, 64, 65, 96, 97, 128, 129):
        assert torch.equal(heads(n), whole[:n]), n
    rows = x.double().view(M, H, K + tail)
    want = torch.einsum("mhk,hnk->mhn", rows[..., :K], w.double())
    if gated:
        want = want * torch.sigmoid(gate.double().view(M, H, N))
    got = whole.double().view(M, H, N + tail)
    room = 2.0 ** -8 * want.abs() + (K * 2.0 ** -24) * torch.einsum("mhk,hnk->mhn", rows[..., :K].abs(), w.double().abs())
    assert bool(((got[..., :N] - want).abs() <= room).all())
    if tail:
        c, s = cos.double()[positions.long()][:, None], sin.double()[positions.long()][:, None]
        t = rows[..., K:]
        a, b = t[..., :rot // 2], t[..., rot // 2:rot]
        turned = torch.cat([a * c - b * s, b * c + a * s, t[..., rot:]], dim=-1)
        assert bool(((got[..., N:] - turned).abs() <= 2.0 ** -8 * turned.abs() + 2.0 ** -22 * (a.abs().max() + b.abs().max())).all())


@pytest.mark.parametrize("K", [64, 128, 192, 256, 320])
@pytest.mark.parametrize("M", [65, 193, 257])
def test_heads_products_in_tall_tiles(M, K):
    """Heads enough for tiles of 128 x 128 (a ring of two stages: K of one, of two and of more, even and odd) have the bits of a few of them,
    which go through tiles of 64 x 128, with a gate and without."""
    from jllm_serve_amd.kernels import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(M + K)
    H, N = 256, 132  # 512 tiles of either kind for each of their rows
    x = torch.randn(M, H * K, device="cuda", generator=gen).bfloat16()
    w = (torch.randn(H, N, K, device="cuda", generator=gen) * K ** -0.5).bfloat16()
    gate = torch.randn(M, H * N, device="cuda", generator=gen).bfloat16()
    plain, gated = ops.latent_heads(x, w), ops.latent_heads(x, w, gate=gate)
    want = torch.einsum("mhk,hnk->mhn", x.double().view(M, H, K), w.double())
    room = 2.0 ** -8 * want.abs() + (K * 2.0 ** -24) * torch.einsum("mhk,hnk->mhn", x.double().abs().view(M, H, K), w.double().abs())
    assert bool(((plain.double().view(M, H, N) - want).abs() <= room).all())
    for h in (0, 137, H - 2):
        at, to = slice(h * K, (h + 2) * K), slice(h * N, (h + 2) * N)
        assert torch.equal(ops.latent_heads(x[:, at].contiguous(), w[h:h + 2].contiguous()), plain[:, to])
        assert torch.equal(ops.latent_heads(x[:, at].contiguous(), w[h:h + 2].contiguous(), gate=gate[:, to].contiguous()), gated[:, to])


@pytest.mark.parametrize("N,K", [(16, 8), (20, 72), (33 * 4, 520), (48, 1096), (36, 2048), (64, 2128)])
def test_grouped_products_of_few_rows(N, K):
    """The experts' products for few rows per expert at the ends of K (whole turns of 512 of a workgroup, parts of one,
    single pieces of 8) and of N, gated and plain, every row map, against float64: sums of K products of bf16 numbers in
    fp32 (an error of K 2^-24 of the sum of magnitudes at most), rounded once where the output is bf16."""
    from jllm_serve_amd.kernels import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    E, top, T = 5, 2, 23
    w, w2 = (torch.randn(E, N, K, device="cuda", generator=gen).bfloat16() for _ in range(2))
    table = torch.rand(T, E, device="cuda", generator=gen).argsort(dim=1)[:, :top].to(torch.int32).contiguous()
    table[:20] = torch.tensor([3, 1], dtype=torch.int32, device="cuda")  # an expert with more rows than one tile holds
    routing = ops.moe_route(None, table, E)
    experts = table.long().reshape(-1)
    x = torch.randn(T, K, device="cuda", generator=gen).bfloat16()
    rows = x.double().repeat_interleave(top, dim=0)
    y, u = (torch.einsum("ak,ank->an", rows, t.double()[experts]) for t in (w, w2))
    room = K * 2.0 ** -24 * torch.einsum("ak,ank->an", rows.abs(), w.double()[experts].abs())
    place = routing.place_of.long()
    out = torch.full((T * top, N), float("nan"), device="cuda")
    ops.moe_gemm(x, w, routing, out=out, in_map=1, out_map=0)
    assert bool(((out[place].double() - y).abs() <= room + 1e-30).all())
    by_assignment = torch.full_like(out, float("nan"))
    ops.moe_gemm(x, w, routing, out=by_assignment, in_map=1, out_map=1)
    assert torch.equal(by_assignment, out[place])
    h = torch.full((T * top, N), float("nan"), device="cuda", dtype=torch.bfloat16)
    ops.moe_gemm(x, w, routing, w2=w2, out=h, in_map=1, out_map=0)
    want = y * torch.sigmoid(y) * u
    scale = (y.abs() + 1.0) * (u.abs() + 1.0) * (1.0 + room.max())
    assert bool(((h[place].double() - want).abs() <= 2.0 ** -8 * want.abs() + 4.0 * room.max() * scale + 2.0 ** -20 * scale).all())


@pytest.mark.parametrize("N,K", [(48, 64), (20, 320), (132, 1024), (36, 1088), (64, 2048), (40, 2368), (16, 4160)])
def test_experts_rows_have_the_same_bits_in_few_and_in_many(N, K):
    """A row's outputs from the tiles of 16 rows (K over the waves of a workgroup, whole turns and parts of one) and from the
    tiles of 128, bit for bit, plain and gated."""
    from jllm_serve_amd.kernels import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    E, top, T = 3, 2, 130
    w, w2 = (torch.randn(E, N, K, device="cuda", generator=gen).bfloat16() for _ in range(2))
    table = torch.rand(T, E, device="cuda", generator=gen).argsort(dim=1)[:, :top].to(torch.int32).contiguous()
    x = (torch.randn(T, K, device="cuda", generator=gen) * K ** -0.5).bfloat16()
    got = []
    for many in (False, True):
        routing = ops.moe_route(None, table, E, many_ok=many)
        assert routing.many == many
        place = routing.place_of.long()
        plain = torch.full((T * top, N), float("nan"), device="cuda")
        ops.moe_gemm(x, w, routing, out=plain, in_map=1, out_map=0)
        pairs = torch.full((T * top, N), float("nan"), device="cuda")
        ops.moe_gemm(x, w, routing, w2=w2, out=pairs, in_map=1, out_map=0)
        got.append((plain[place], pairs[place]))
    assert bool(torch.isfinite(got[0][0]).all())
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("K", [64, 128, 192, 320, 704])
@pytest.mark.parametrize("N", [64, 132, 260])
def test_experts_tiles_at_their_edges(N, K):
    """Experts with no row, one, one short of a tile, a whole tile, one beyond it and two tiles and one, K of one stage, of the ring's two
    and of even and odd numbers beyond: gathered rows and rows by place, plain and gated, against float64."""
    from jllm_serve_amd.kernels import ops
    gen = torch.Generator(device="cuda")
    gen.manual_seed(N + K)
    counts = [0, 1, 127, 128, 129, 257]
    E, T = len(counts), sum(counts)
    w, w2 = ((torch.randn(E, N, K, device="cuda", generator=gen) * K ** -0.5).bfloat16() for _ in range(2))
    experts = torch.repeat_interleave(torch.arange(E, device="cuda"), torch.tensor(counts, device="cuda"))[torch.randperm(T, device="cuda", generator=gen)]
    routing = ops.moe_route(None, experts.to(torch.int32).view(T, 1).contiguous(), E, many_ok=True)
    assert routing.many
    x = torch.randn(T, K, device="cuda", generator=gen).bfloat16()
    y, u = (torch.einsum("ak,ank->an", x.double(), t.double()[experts]) for t in (w, w2))
    room = K * 2.0 ** -24 * torch.einsum("ak,ank->an", x.double().abs(), w.double()[experts].abs())
    place = routing.place_of.long()
    by_place = torch.empty_like(x)
    by_place[place] = x
    for a, in_map in ((x, 1), (by_place, 0)):
        out = torch.full((T, N), float("nan"), device="cuda")
        ops.moe_gemm(a, w, routing, out=out, in_map=in_map, out_map=0)
        assert bool(((out[place].double() - y).abs() <= room + 1e-30).all())
        h = torch.full((T, N), float("nan"), device="cuda", dtype=torch.bfloat16)
        ops.moe_gemm(a, w, routing, w2=w2, out=h, in_map=in_map, out_map=0)
        want = y * torch.sigmoid(y) * u
        scale = (y.abs() + 1.0) * (u.abs() + 1.0)
        assert bool(((h[place].double() - want).abs() <= 2.0 ** -8 * want.abs() + 4.0 * room.max() * scale + 2.0 ** -20 * scale).all())


@pytest.mark.parametrize("dtype, fast", [("float32", False), ("bfloat16", True), ("bfloat16", False)])
@pytest.mark.parametrize("H, R, Dr, page", [(4, 32, 16, 8), (5, 48, 8, 16), (16, 64, 32, 32), (40, 16, 16, 4), (3, 24, 6, 8)])
def test_attention_kernels_on_crafted_keys(dtype, fast, H, R, Dr, page):
    """One key far back carries a value unlike all others and a score that dominates. The query rows are placed so
    that this key is the window's oldest key, one beyond it, at a page's first and last place, and hundreds of keys
    away without a window; as rows of a long portion and as single rows of other requests. A kernel that is one key
    off at an edge, or drops the sink, is off by the size of the values."""
    from jllm_serve_amd.kernels import ops
    from jllm_serve_amd.parts.latent_attention import LatentStepPlanner, TILE_ROWS
    t = torch.float32 if dtype == "float32" else torch.bfloat16
    Dk = R + Dr
    g = torch.Generator().manual_seed(H * 1000 + R)
    L = 613
    hot = 3 * page + page - 1 if page > 4 else 131  # the last place of a page
    rows = (torch.randn(L, Dk, generator=g) * 0.3).to(t).double()
    direction = torch.nn.functional.normalize(torch.randn(Dk, generator=g), dim=0).to(t).double()
    rows[hot] = (direction * 6.0 + rows[hot]).to(t).double()
    rows[hot, :R] += 2.0  # its value stands out
    rows = rows.to(t).double()
    sink = torch.randn(H, generator=g) * 2 + 1.0
    for window in (0, 37, 64, 300):
        # requests: 0 = one long portion of all rows from position 0; then single rows of further requests that hold the
        # same keys, placed at the edges
        edges = sorted({hot, hot + 1, hot + page, L - 1} | ({hot + window - 1, hot + window, hot + window + 1} if window else {400}))
        edges = [p for p in edges if p < L]
        n_req = 1 + len(edges)
        qa = (torch.randn(L + len(edges), H, Dk, generator=g) * 0.3 + direction * 2.5).to(t)
        q_pos = torch.cat([torch.arange(L), torch.tensor(edges)])
        want = _attend_plain(qa.double(), rows, R, window, 0.9, sink.double(), q_pos)
        # the far key decides rows that see it: the test is blind otherwise
        sees = (q_pos >= hot) & ((q_pos - hot < window) if window else torch.ones_like(q_pos, dtype=torch.bool))
        assert want[sees][..., :R].mean() > 1.0 and want[~sees][..., :R].mean() < 0.5
        width = -(-L // page)
        pages = list(range(n_req * width))
        random.Random(window).shuffle(pages)
        table = torch.tensor(pages, dtype=torch.int32).view(n_req, width)
        cache = torch.full((n_req * width, page, Dk), float("nan"), dtype=t)  # a key read from a wrong place poisons the row
        for r in range(n_req):
            n = L if r == 0 else edges[r - 1] + 1
            for p0 in range(0, n, page):
                k = min(page, n - p0)
                cache[table[r, p0 // page], :k] = rows[p0:p0 + k].to(t)
        row_req = torch.cat([torch.zeros(L, dtype=torch.int32), torch.arange(1, n_req, dtype=torch.int32)])
        runs = [(0, r, min(TILE_ROWS, L - r), r) for r in range(0, L, TILE_ROWS)] + [(1 + i, L + i, 1, p) for i, p in enumerate(edges)]
        meta = {"tiles_dev": torch.tensor(runs, dtype=torch.int32).flatten().to(DEV), "n_tiles": len(runs)} if fast else None
        ops.reset_stats()
        out = ops.latent_attention(qa.view(-1, H * Dk).to(DEV), cache.to(DEV), table.to(DEV), row_req.to(DEV),
                                   q_pos.to(torch.int32).to(DEV), H, R, window, 0.9, sink.to(DEV), meta=meta,
                                   exact=dtype == "float32")
        takes = R % 16 == 0 and Dk % 8 == 0  # what the matrix-core kernel takes; other sizes fall to the general kernel
        if fast:
            assert ops.stats()["ran"].get("jllm_latent_attention_bf16", 0) == (1 if takes else 0), ops.stats()
        got = out.view(-1, H, R).double().cpu()
        assert torch.isfinite(got).all(), f"window {window}: a row read a place that holds no key"
        err = (got - want).abs().amax(dim=(1, 2))
        tol = 1e-4 if dtype == "float32" else 4e-2
        bad = (err > tol).nonzero().flatten().tolist()
        assert not bad, f"window {window}: rows at positions {[int(q_pos[i]) for i in bad[:8]]} differ by up to {float(err.max())}"
        if fast:  # the single rows alone, as a decode step: their keys are cut into ranges over several workgroups
            n1 = len(edges)
            meta1 = {"tiles_dev": torch.tensor([(1 + i, i, 1, p) for i, p in enumerate(edges)], dtype=torch.int32).flatten().to(DEV),
                     "n_tiles": n1, "single_rows": True, "max_context": L}
            assert ops._latent_split(n1, H, window, L)[0] > 0 or window in (37, 64)
            out1 = ops.latent_attention(qa[L:].reshape(n1, H * Dk).to(DEV), cache.to(DEV), table.to(DEV), row_req[L:].to(DEV),
                                        q_pos[L:].to(torch.int32).to(DEV), H, R, window, 0.9, sink.to(DEV), meta=meta1)
            err1 = (out1.view(n1, H, R).double().cpu() - want[L:]).abs().amax(dim=(1, 2))
            assert float(err1.max()) <= tol, f"window {window}: single rows at {edges} differ by {err1.tolist()}"
        if window == 0:  # without the sink the same rows are far off: the sink is not lost in the noise
            no_sink = _attend_plain(qa.double(), rows, R, window, 0.9, None, q_pos)
            assert (no_sink - want).abs().max() > 0.3


@pytest.mark.parametrize("H, R, Dk, window", [(16, 512, 576, 0), (16, 512, 576, 130), (3, 144, 168, 70), (40, 496, 520, 0), (7, 128, 256, 64), (6, 80, 104, 50),
                                              (2, 128, 128, 0)])
def test_latent_attention_of_runs_of_rows(H, R, Dk, window):
    """Portions of prompts in runs of 1 to 16 rows that begin at any position (keys end one below, at and one beyond a
    block of 64; a single row beside them), rows whose entries are no multiple of 32 or 64, latents whose last waves have no
    part; every sum from the definition in 64 bits."""
    from jllm_serve_amd.kernels import ops
    g = torch.Generator().manual_seed(R + H + window)
    page, spans = 16, [(0, 33), (58, 6), (63, 1), (64, 1), (200, 63), (257, 1)]  # (first position, rows) of each request
    width = 24
    n_req = len(spans)
    cache = torch.full((n_req * width, page, Dk), float("nan"), dtype=torch.bfloat16)
    table = torch.randperm(n_req * width, generator=g).to(torch.int32).view(n_req, width)
    sink = torch.randn(H, generator=g)
    rows, runs, pos, req, want, room = [], [], [], [], [], []
    scale = 1.5 * Dk ** -0.5
    for r, (p0, n) in enumerate(spans):
        keys = torch.randn(p0 + n, Dk, generator=g).bfloat16()
        for k in range(0, p0 + n, page):
            part = keys[k:k + page]
            cache[int(table[r, k // page]), :len(part)] = part
        q = torch.randn(n, H, Dk, generator=g).bfloat16()
        runs += [(r, len(pos) + i, min(16, n - i), p0 + i) for i in range(0, n, 16)]
        rows.append(q)
        at = torch.arange(p0, p0 + n)
        pos += at.tolist()
        req += [r] * n
        z = torch.einsum("nhd,kd->nhk", q.double(), keys.double()) * scale
        key = torch.arange(p0 + n)
        seen = (key <= at[:, None]) & ((key > at[:, None] - window) if window else torch.ones_like(key, dtype=torch.bool))
        z = z.masked_fill(~seen[:, None], -torch.inf)
        p = torch.softmax(torch.cat([z, sink.double().expand(n, H)[..., None]], dim=2), dim=2)[..., :-1]
        want.append(p @ keys[:, :R].double())
        # a score: Dk products' fp32 sum, in any order, and its part in exp; the probabilities and the result as bf16
        size = torch.einsum("nhd,kd->nhk", q.double().abs(), keys.double().abs()).amax(dim=2, keepdim=True) * scale
        room.append((2.0 ** -9 + 2.0 * Dk * 2.0 ** -24 * size + 2.0 ** -18) * (p @ keys[:, :R].double().abs()) + 2.0 ** -8 * want[-1].abs())
    meta = {"tiles_dev": torch.tensor(runs, dtype=torch.int32).flatten().to(DEV), "n_tiles": len(runs)}
    ops.reset_stats()
    got = ops.latent_attention(torch.cat(rows).view(-1, H * Dk).to(DEV), cache.to(DEV), table.to(DEV), torch.tensor(req, dtype=torch.int32, device=DEV),
                               torch.tensor(pos, dtype=torch.int32, device=DEV), H, R, window, scale, sink.to(DEV), meta=meta)
    assert ops.stats()["ran"] == {"jllm_latent_attention_bf16": 1}
    assert bool(((got.view(-1, H, R).double().cpu() - torch.cat(want)).abs() <= torch.cat(room)).all())


@pytest.mark.parametrize("H, R, Dk", [(16, 512, 576), (40, 512, 576), (5, 64, 128), (70, 128, 256), (16, 512, 568)])
@pytest.mark.parametrize("window", [0, 100, 300])
def test_latent_attention_of_single_rows_of_whole_sizes(H, R, Dk, window):
    """Single rows at the sizes whose loops carry no condition (and one entry group short of them), in ranges of one block and uncut:
    keys that end one below, at and one beyond a block or a range, places without keys hold NaN; the definition in 64 bits."""
    from jllm_serve_amd.kernels import ops
    g = torch.Generator().manual_seed(H + R + window)
    page, width, pos = 16, 48, [0, 62, 63, 64, 255, 256, 699, 767]
    n = len(pos)
    assert ops._latent_split(n, H, window, width * page) == ((0, 1) if window == 100 else (64, 6) if window == 300 else (64, 13))
    cache = torch.full((n * width, page, Dk), float("nan"), dtype=torch.bfloat16)
    table = torch.randperm(n * width, generator=g).to(torch.int32).view(n, width)
    q, sink, scale = torch.randn(n, H, Dk, generator=g).bfloat16(), torch.randn(H, generator=g), 1.5 * Dk ** -0.5
    want, room = [], []
    for r, at in enumerate(pos):
        keys = torch.randn(at + 1, Dk, generator=g).bfloat16()
        for k in range(0, at + 1, page):
            part = keys[k:k + page]
            cache[int(table[r, k // page]), :len(part)] = part
        keys = keys[max(0, at + 1 - window) if window else 0:].double()
        z = q[r].double() @ keys.T * scale
        p = torch.softmax(torch.cat([z, sink.double()[:, None]], dim=1), dim=1)[:, :-1]
        want.append(p @ keys[:, :R])
        # a score: Dk products' fp32 sum, in any order, and its part in exp; the probabilities and the result as bf16
        size = (q[r].double().abs() @ keys.abs().T).amax(dim=1, keepdim=True) * scale
        room.append((2.0 ** -9 + 2.0 * Dk * 2.0 ** -24 * size + 2.0 ** -18) * (p @ keys[:, :R].abs()) + 2.0 ** -8 * want[-1].abs())
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    meta = {"tiles_dev": i32([(i, i, 1, p) for i, p in enumerate(pos)]).flatten(), "n_tiles": n, "single_rows": True, "max_context": width * page}
    got = ops.latent_attention(q.view(n, -1).to(DEV), cache.to(DEV), table.to(DEV), i32(list(range(n))), i32(pos), H, R, window, scale, sink.to(DEV), meta=meta)
    assert bool(((got.view(n, H, R).double().cpu() - torch.stack(want)).abs() <= torch.stack(room)).all())


@pytest.mark.parametrize("H, R, Dk, window, single_runs", [(40, 512, 576, 0, False), (40, 144, 168, 90, False), (17, 128, 256, 33, False),
                                                           (16, 512, 576, 0, True), (16, 512, 576, 70, True), (3, 96, 128, 0, True), (20, 64, 96, 0, False)])
def test_latent_attention_gives_a_row_the_same_bits_in_runs_and_alone(H, R, Dk, window, single_runs):
    """A row's result as a single row of its step and in a run of a portion, bit for bit: with more than 16 heads in runs of up
    to 16 rows; with up to 16, where a row alone keeps four sums, in runs of one row. Keys grow along the context, so that
    the running maxima move in every place of a block, and one request has equal keys."""
    from jllm_serve_amd.kernels import ops
    g = torch.Generator().manual_seed(H + Dk + window)
    page, spans = 16, [(0, 100), (58, 6), (63, 1), (100, 130), (250, 5), (0, 1)]
    width = 16
    cache = torch.randn(len(spans) * width, page, Dk, generator=g)
    table = torch.randperm(len(spans) * width, generator=g).to(torch.int32).view(len(spans), width)
    for r in range(len(spans)):
        cache[table[r].long()] *= (torch.arange(width * page).view(width, page, 1) / 60.0) if r != 3 else 1.0
    cache = cache.bfloat16().to(DEV)
    pos = [p for p0, n in spans for p in range(p0, p0 + n)]
    req = [r for r, (p0, n) in enumerate(spans) for _ in range(n)]
    q = (torch.randn(len(pos), H * Dk, generator=g) * 2).bfloat16().to(DEV)
    sink = torch.randn(H, generator=g).to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    rows = [(req[i], i, 1, pos[i]) for i in range(len(pos))]
    runs, at = rows, 0
    if not single_runs:
        runs = []
        for r, (p0, n) in enumerate(spans):
            runs += [(r, at + i, min(16, n - i), p0 + i) for i in range(0, n, 16)]
            at += n

    def attend(tiles, **facts):
        return ops.latent_attention(q, cache, table.to(DEV), i32(req), i32(pos), H, R, window, Dk ** -0.5, sink,
                                    meta={"tiles_dev": i32(tiles).flatten(), "n_tiles": len(tiles), **facts})

    assert ops._latent_split(len(rows), H, window, 255) == (0, 1)
    alone = attend(rows, single_rows=True, max_context=255)
    assert bool(torch.isfinite(alone).all())
    assert torch.equal(attend(runs), alone)


@pytest.mark.parametrize("H", [3, 16, 40])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_latent_attention_of_runs_keeps_infinities_with_the_rows_that_see_them(H, bad):
    """A cached entry that is no finite number, behind some of a run's rows and out of the window of others: only the rows
    that see it may feel it, and those do."""
    from jllm_serve_amd.kernels import ops
    g = torch.Generator().manual_seed(H)
    R, Dk, page, n, window = 64, 96, 16, 150, 40
    cache = torch.randn(16, page, Dk, generator=g).bfloat16()
    table = torch.randperm(16, generator=g).to(torch.int32).view(1, 16)
    at = torch.arange(n)
    q = torch.randn(n, H, Dk, generator=g).bfloat16()
    keys = cache[table[0].long()].view(-1, Dk)[:n].double()
    runs = [(0, i, min(16, n - i), i) for i in range(0, n, 16)]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    for place in (1, 35, 63, 70, 149):
        spoiled = cache.clone()
        spoiled[int(table[0, place // page]), place % page, 5] = bad
        got = ops.latent_attention(q.view(n, -1).to(DEV), spoiled.to(DEV), table.to(DEV), torch.zeros(n, dtype=torch.int32, device=DEV),
                                   i32(at.tolist()), H, R, window, Dk ** -0.5, None,
                                   meta={"tiles_dev": i32(runs).flatten(), "n_tiles": len(runs)}).cpu().double().view(n, H, R)
        z = torch.matmul(q.double(), keys.T) * Dk ** -0.5
        z = z.masked_fill(((at[None] > at[:, None]) | (at[None] <= at[:, None] - window))[:, None], -torch.inf)
        p = torch.softmax(z, dim=2)
        want = torch.matmul(p, keys[:, :R])
        room = (2.0 ** -8 + 2.0 ** -18) * torch.matmul(p, keys[:, :R].abs()) + 2.0 ** -8 * want.abs()
        sees = (at >= place) & (at < place + window)
        assert bool(((got - want).abs() <= room)[~sees].all()), place
        assert not bool(torch.isfinite(got[sees]).all(dim=2).any()), place


@pytest.mark.parametrize("Dk", [576, 584, 640])
def test_latent_rows_too_long_for_the_matrix_core_kernel_take_the_general_one(Dk):
    """Cached rows at the longest that the matrix-core kernel takes and beyond, as a run of a portion and as single rows."""
    from jllm_serve_amd.kernels import ops
    g = torch.Generator().manual_seed(Dk)
    H, R, page, n = 5, 512, 16, 40
    cache = torch.randn(4, page, Dk, generator=g).bfloat16()
    q = torch.randn(n, H, Dk, generator=g).bfloat16()
    table = torch.tensor([[2, 0, 3, 1]], dtype=torch.int32)
    keys = cache[table[0].long()].view(-1, Dk)[:n].double()
    at = torch.arange(n)
    z = (torch.matmul(q.double(), keys.T) * Dk ** -0.5).masked_fill((at[None] > at[:, None])[:, None], -torch.inf)
    p = torch.softmax(z, dim=2)
    want, room = torch.matmul(p, keys[:, :R]), 2.0 ** -8 * torch.matmul(p, keys[:, :R].abs())
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    runs, rows = [(0, i, min(16, n - i), i) for i in range(0, n, 16)], [(0, i, 1, i) for i in range(n)]
    for tiles, facts in ((runs, {}), (rows, {"single_rows": True, "max_context": n})):
        ops.reset_stats()
        got = ops.latent_attention(q.view(n, -1).to(DEV), cache.to(DEV), table.to(DEV), torch.zeros(n, dtype=torch.int32, device=DEV), i32(at.tolist()),
                                   H, R, 0, Dk ** -0.5, None, meta={"tiles_dev": i32(tiles).flatten(), "n_tiles": len(tiles), **facts})
        stats = ops.stats()
        assert bool(stats["general"]) == (Dk > 576) and bool(stats["ran"]) == (Dk <= 576), stats
        assert bool(((got.view(n, H, R).double().cpu() - want).abs() <= 2.0 ** -8 * want.abs() + room).all())


# ------------------------------------------------------------------------------------------------ replays


def _replay(model, trace, page, shuffle=None):
    from jllm_serve_amd.engine.trace import TraceRunner
    tr = TraceRunner(None, None, trace.peak, page_size=page, max_live=4, shuffle_free=shuffle, model=model)
    out = {}
    for rec in trace.steps:
        logits = tr.step(rec)
        if rec["step"] in trace.rows:
            got = logits.float().cpu()
            for (rid, p), row in zip(trace.rows[rec["step"]], got):
                out[(rid, p)] = row
    tr.runner.cache.check()
    assert not tr.runner.cache.requests and all(g.pool.used_pages == 0 for g in tr.runner.cache.groups)
    return out, tr.runner


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name", ["MA", "MB", "MC"])
def test_replays_match_plain_and_each_other(name, dtype, miforax_folders, plain_logits):
    """Whole prompts, the last tokens one by one (captured steps in bfloat16), portions down to two tokens, and mixed
    batches of up to four requests on a pool exactly as large as the busiest step with free pages in random order."""
    from jllm_serve_amd.engine import load_model
    page = mt.CONFIGS[name][2]
    model = load_model(miforax_folders[name], dtype, torch.device(DEV), max_positions=512)
    reqs = {f"r{n}": mt.prompt(name, n, seed=1) for n in (1, 2, 9, 23, 41, 70, 133)}
    want = {(rid, p): row for rid, toks in reqs.items() for p, row in enumerate(plain_logits(name, toks))}
    traces = {}
    for kind in ("whole", "tail", "portions", "mixed"):
        tr = replay.Trace(page)
        if kind == "mixed":
            replay.mixed(tr, reqs, seed=3)
        else:
            for rid, toks in reqs.items():
                {"whole": replay.whole, "tail": replay.tail_one_by_one, "portions": replay.portions}[kind](tr, rid, toks)
        traces[kind] = tr
    got = {}
    for kind, tr in traces.items():
        got[kind], runner = _replay(model, tr, page, shuffle=7 if kind == "mixed" else None)
        assert set(got[kind]) == set(want)
        # against the tolerance at the size of the request's logits (a single row's largest logit may be small)
        scale = {rid: plain_logits(name, toks) for rid, toks in reqs.items()}
        worst = max(float((got[kind][k].double() - want[k]).abs().max()) / mt.tolerance(dtype, scale[k[0]]) for k in want)
        assert worst <= 1.0, f"{kind}: {worst} of the tolerance"
        if kind == "tail" and dtype == "bfloat16":
            assert runner.graphs is not None and runner.graphs.replays > 0, "single tokens did not go through captured steps"
    if dtype == "float32":  # cutting and batching change nothing but the last bits
        for kind in ("tail", "portions", "mixed"):
            d = max(float((got[kind][k] - got["whole"][k]).abs().max()) for k in want)
            assert d <= 2e-5, f"{kind} differs from whole prompts by {d}"


@pytest.mark.parametrize("name, dtype", [("MA", "float32"), ("MB", "bfloat16"), ("MA", "bfloat16")])
def test_long_decoding_lets_every_window_pass_over_decoded_tokens(name, dtype, miforax_folders, plain_logits):
    from jllm_serve_amd.engine import build_runner, load_model
    from jllm_serve_amd.engine.step import StepEntry
    page = mt.CONFIGS[name][2]
    model = load_model(miforax_folders[name], dtype, torch.device(DEV), max_positions=256)
    runner = build_runner(model, page_size=page, pool_tokens=256, max_requests=2)
    toks = mt.prompt(name, 170, seed=9)
    want = plain_logits(name, toks)
    got = [runner.step([StepEntry("d", toks[:12], list(range(12)))]).float().cpu()]
    for i in range(12, len(toks)):
        got.append(runner.step([StepEntry("d", toks[i:i + 1], [0])]).float().cpu())
    given_back = runner.cache.stats()["window_pages_given_back"]
    runner.finish("d")
    close(torch.cat(got), want, dtype, "170 positions, 158 of them decoded one by one")
    assert given_back > 0, "no window gave a page back"


def test_greedy_generation_through_the_engine(miforax_folders):
    from jllm_serve_amd.engine import Engine, SchedulerConfig, build_runner, load_model
    from jllm_serve_amd.sampling import SamplingParams
    cfg, _, page = mt.CONFIGS["MA"]
    w = mt.load_weights(miforax_folders["MA"])
    prompts = [mt.prompt("MA", n, seed=2) for n in (5, 17, 33, 2)]
    want = [P.greedy(cfg, w, p, 12) for p in prompts]
    for dtype in ("float32", "bfloat16"):
        model = load_model(miforax_folders["MA"], dtype, torch.device(DEV), max_positions=128)
        runner = build_runner(model, page_size=page, pool_tokens=256, max_requests=3)  # four requests, three places
        eng = Engine(runner, SchedulerConfig(max_batch_tokens=24, prefill_chunk=16, max_positions=128), eos_token_ids=())
        res = eng.generate(prompts, SamplingParams.greedy_params(max_tokens=12))
        if dtype == "float32":
            assert [r.tokens for r in res] == want
        else:
            agree = sum(a == b for r, x in zip(res, want) for a, b in zip(r.tokens, x))
            assert all(r.tokens[0] == x[0] for r, x in zip(res, want)) and agree >= 36, f"bfloat16 agrees on {agree}/48 tokens"


def test_replay_program_and_command_line(miforax_folders, plain_logits, tmp_path):
    """bin/trace_run picks the model class by config.json; the command line generates from the same folder."""
    import subprocess
    import sys
    tr = replay.Trace(64)
    reqs = {"a": mt.prompt("MA", 21, seed=5), "b": mt.prompt("MA", 40, seed=6)}
    replay.mixed(tr, reqs, seed=1)
    got = replay.run(miforax_folders["MA"], "float32", tr, str(tmp_path / "out"), page_size=8)
    for step, rows in tr.rows.items():
        arr = got[step].reshape(len(rows), -1)
        for (rid, p), row in zip(rows, arr):
            ref = plain_logits("MA", reqs[rid])[p]
            assert float((torch.from_numpy(row.copy()).double() - ref).abs().max()) <= mt.tolerance("float32", ref)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, os.path.join(root, "bin", "jllm"), "run", "--model", miforax_folders["MA"], "--dtype", "float32",
                        "--prompt", " ".join(map(str, reqs["a"])), "--max-tokens", "6", "--temp", "0", "--json", "--ctx", "128",
                        "--ignore-eos"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    out = json.loads(r.stdout.strip().splitlines()[-1])
    assert out["tokens"] == P.greedy(mt.MF_A, mt.load_weights(miforax_folders["MA"]), reqs["a"], 6)
