"""The work that is measured: steps of whole models through the engine's step function.

A case is a model (a family, one of the sizes that ``bench.py`` names, a run type) and what one pass asks of it:

* ``decode``: every request holds its prompt already and brings one token; the pass is one step and forgets the
  tokens again (``cache.truncate``), so that every pass does the same work;
* ``prefill``: one step of whole prompts, whose last rows' logits are wanted; the requests end with the pass;
* ``mixed``: one step with a portion of a long prompt beside the single rows of decoding requests;
* ``serve``: prompts in one step, then a few steps of one token per request, then the requests end.

The requests of a case have lengths spread over ``shortest`` .. ``longest`` by a fixed rule; token ids and weights come
from the seed. Weights are random at the scales that trained models keep: a product has the variance of its input, what a
sublayer adds to the stream is scaled by 1 / sqrt(sublayers) so that no layer drowns the ones before it, gains are
1 + N(0, 0.1), and the recurrent layers' decays and taps lie in the usual ranges. Tokens are given rather than sampled:
which token comes next does not change what a step costs, and outputs stay comparable where two logits are close.
"""
import math
import os
import sys
import zlib

import torch

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))

from jllm_serve_amd.config import parse_config  # noqa: E402
from jllm_serve_amd.engine import StepEntry, build_model, build_runner  # noqa: E402

PAGE = 16
POSITIONS = 8192  # positions a request may hold
PLACES = 64  # requests that may run at once
PORTION = 2048  # rows of a prompt per step while a state is prepared

QWEN3 = {  # layers, width, heads, kv heads, head size, feed-forward
    "0.6b": (28, 1024, 16, 8, 128, 3072),
    "1.7b": (28, 2048, 16, 8, 128, 6144),
    "4b": (36, 2560, 32, 8, 128, 9728),
    "8b": (36, 4096, 32, 8, 128, 12288),
    "14b": (40, 5120, 40, 8, 128, 17408),
    "32b": (64, 5120, 64, 8, 128, 25600),
}
QWEN3_VOCAB = 151936
QWEN3_BASE = 1e6
VOCAB = 32768  # of the other two families, as the benchmark has them
LAYERS = 4
MIFORAX = {
    "2k": dict(width=2048, heads=16, q_rank=768, window=1024, ff=8192, experts=32, top=4, expert_ff=1024, shared_ff=4096),
    "4k": dict(width=4096, heads=32, q_rank=1536, window=4096, ff=12288, experts=64, top=6, expert_ff=1536, shared_ff=3072),
}
LATENT = dict(dim=128, rot=64, vdim=128, kv_rank=512)
KEBEPEL = {
    "2k": dict(width=2048, heads=16, kv_heads=8, d_heads=8, r_heads=16, r_kv_heads=8, ff=8192),
    "4k": dict(width=4096, heads=32, kv_heads=8, d_heads=16, r_heads=32, r_kv_heads=16, ff=12288),
}
WIDE = dict(dim=128, vdim=128, d_kv_heads=4, d_vdim=256, conv=4)
YARN = {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}
EPS = 1e-6


# ------------------------------------------------------------------------------------------------ the cases


def listed():
    return [
        # a short chat with the smallest model: launches and latencies, not bytes
        dict(name="chat_0.6b", family="qwen3", size="0.6b", dtype="bf16", kind="decode", requests=1, shortest=300, longest=300),
        # the headline: decoding at the 8B shape, alone, as a small batch and as a full one
        dict(name="decode_8b_1", family="qwen3", size="8b", dtype="bf16", kind="decode", requests=1, shortest=2048, longest=2048),
        dict(name="decode_8b_8", family="qwen3", size="8b", dtype="bf16", kind="decode", requests=8, shortest=900, longest=2500),
        dict(name="decode_8b_64", family="qwen3", size="8b", dtype="bf16", kind="decode", requests=64, shortest=250, longest=1000),
        # a few long conversations (documents, code): the cache is half of what a step reads
        dict(name="long_4b_4", family="qwen3", size="4b", dtype="bf16", kind="decode", requests=4, shortest=6100, longest=8000),
        # the headline's other half: one prompt
        dict(name="prefill_8b_2048", family="qwen3", size="8b", dtype="bf16", kind="prefill", requests=1, shortest=2048, longest=2048),
        # a short prompt to the smallest model: the time to its first token
        dict(name="prefill_0.6b_487", family="qwen3", size="0.6b", dtype="bf16", kind="prefill", requests=1, shortest=487, longest=487),
        # prompts of any lengths that arrive together at a larger model
        dict(name="prefill_14b_ragged", family="qwen3", size="14b", dtype="bf16", kind="prefill", requests=3, shortest=709, longest=2051),
        # what a busy server runs most: new prompt rows beside the requests that decode
        dict(name="mixed_8b", family="qwen3", size="8b", dtype="bf16", kind="mixed", requests=20, shortest=300, longest=1400,
             portion=611, behind=1024),
        # the run type whose every sum is in 32 bits: prompts and a few tokens
        dict(name="float32_0.6b", family="qwen3", size="0.6b", dtype="fp32", kind="serve", requests=3, shortest=90, longest=402, tokens=6),
        # latent attention with routed experts, and attention beside a delta rule: prompts and tokens
        dict(name="miforax_2k", family="miforax", size="2k", dtype="bf16", kind="serve", requests=5, shortest=130, longest=1211, tokens=16),
        dict(name="kebepel_2k", family="kebepel", size="2k", dtype="bf16", kind="serve", requests=4, shortest=150, longest=1390, tokens=16),
    ]


def draw(rng):
    def spread(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    def lengths(n, low, high, most):
        """A longest and a shortest length: together no more than ``most`` rows."""
        b = min(spread(low, high), max(low, most // n))
        return dict(requests=n, shortest=max(low, int(b * rng.uniform(0.25, 1.0))), longest=b)

    kind = rng.choice(["decode"] * 7 + ["prefill"] * 4 + ["mixed"] * 3 + ["float32"] * 2 + ["miforax"] * 2 + ["kebepel"] * 2)
    if kind == "decode":
        size = rng.choice(list(QWEN3))
        most = {"0.6b": 60000, "1.7b": 60000, "4b": 40000, "8b": 36000, "14b": 18000, "32b": 8000}[size]
        return dict(family="qwen3", size=size, dtype="bf16", kind=kind, **lengths(spread(1, 64), 17, 8000, most))
    if kind == "prefill":
        size = rng.choice(["0.6b", "1.7b", "4b", "8b", "14b"])
        n = rng.choice([1, 1, 1, 2, 3, 5, 8])
        return dict(family="qwen3", size=size, dtype="bf16", kind=kind, **lengths(n, 20, 4096, 4096))
    if kind == "mixed":
        size = rng.choice(["0.6b", "1.7b", "4b", "8b", "14b"])
        return dict(family="qwen3", size=size, dtype="bf16", kind=kind, portion=spread(24, 2048), behind=rng.choice([0, spread(16, 4096)]),
                    **lengths(spread(2, 48), 20, 4000, 16000))
    if kind == "float32":
        return dict(family="qwen3", size=rng.choice(["0.6b", "0.6b", "1.7b"]), dtype="fp32", kind="serve", tokens=rng.randint(2, 8),
                    **lengths(rng.randint(1, 8), 20, 1000, 1000))
    return dict(family=kind, size=rng.choice(["2k", "2k", "4k"]), dtype="bf16", kind="serve", tokens=rng.randint(4, 24),
                **lengths(spread(1, 24), 20, 2048, 4096))


def lengths_of(case):
    """The requests' lengths: the first is the longest, the others lie spread between the two bounds."""
    a, b = case["shortest"], case["longest"]
    return [b] + [a + int((b - a) * (i * 0.6180339887 % 1.0)) for i in range(1, case["requests"])]


# ------------------------------------------------------------------------------------------------ models


def config_of(case):
    """The config.json of the case's model."""
    if case["family"] == "qwen3":
        L, d, H, G, hd, F = QWEN3[case["size"]]
        return dict(model_type="qwen3", architectures=["Qwen3ForCausalLM"], num_hidden_layers=L, hidden_size=d, num_attention_heads=H,
                    num_key_value_heads=G, head_dim=hd, intermediate_size=F, vocab_size=QWEN3_VOCAB, rope_theta=QWEN3_BASE,
                    rms_norm_eps=EPS, tie_word_embeddings=False, max_position_embeddings=POSITIONS)
    if case["family"] == "miforax":
        z, y = MIFORAX[case["size"]], LATENT
        mixer = {"heads": z["heads"], "dim": y["dim"], "rot_dim": y["rot"], "vdim": y["vdim"], "q_rank": z["q_rank"],
                 "kv_rank": y["kv_rank"], "scale": (y["dim"] + y["rot"]) ** -0.5, "mask": {"size": z["window"]},
                 "rot": {"base": 1e6, "dims": y["rot"], "scaling": YARN}}
        dense = {"kind": "dense", "ff": z["ff"]}
        moe = {"kind": "moe", "router": {"experts": z["experts"], "top": z["top"]}, "expert": {"ff": z["expert_ff"], "limit": 7.0},
               "shared": {"ff": z["shared_ff"], "limit": 7.0}}
        return {"architecture": "Miforax", "vocab": VOCAB, "width": z["width"], "norm": {"eps": EPS}, "embedding": {"scale": 1.0},
                "max_positions": POSITIONS,
                "layers": [{"type": "latent_attention", "mixer": mixer, "mlp": moe if i % 2 else dense} for i in range(LAYERS)]}
    z, y = KEBEPEL[case["size"]], WIDE
    left = {"heads": z["heads"], "kv_heads": z["kv_heads"], "dim": y["dim"], "vdim": y["vdim"], "scale": y["dim"] ** -0.5,
            "softcap": 30.0, "rot": {"base": 1e6, "dims": y["dim"], "scaling": YARN}}
    right = {"heads": z["r_heads"], "kv_heads": z["r_kv_heads"], "dim": y["dim"], "vdim": y["vdim"], "conv": y["conv"]}
    par = {"type": "parallel", "mixer": {"left": left, "right": right, "left_scale": 1.0, "right_scale": 1.0}, "mlp": {"kind": "dense", "ff": z["ff"]}}
    att = {"type": "attention", "mixer": {"heads": z["d_heads"], "kv_heads": y["d_kv_heads"], "dim": y["dim"], "vdim": y["d_vdim"],
                                          "scale": y["dim"] ** -0.5, "diff": 0.2, "q_temp": {"coef": 0.1, "every": 256}},
           "mlp": {"kind": "dense", "ff": z["ff"]}}
    return {"architecture": "Kebepel", "vocab": VOCAB, "width": z["width"], "norm": {"eps": EPS}, "max_positions": POSITIONS,
            "layers": [att if i % 2 else par for i in range(LAYERS)]}


def tensors_of(case):
    """name -> (shape, how it is filled) of every tensor of the case's model."""
    w = {}
    if case["family"] == "qwen3":
        L, d, H, G, hd, F = QWEN3[case["size"]]
        w["model.embed_tokens.weight"], w["lm_head.weight"] = ((QWEN3_VOCAB, d), "embedding"), ((QWEN3_VOCAB, d), "matrix")
        w["model.norm.weight"] = ((d,), "gain")
        for i in range(L):
            p = "model.layers.%d." % i
            w[p + "input_layernorm.weight"] = w[p + "post_attention_layernorm.weight"] = ((d,), "gain")
            for n, rows in (("q", H * hd), ("k", G * hd), ("v", G * hd)):
                w[p + "self_attn.%s_proj.weight" % n] = ((rows, d), "matrix")
            w[p + "self_attn.o_proj.weight"] = ((d, H * hd), "out")
            w[p + "self_attn.q_norm.weight"] = w[p + "self_attn.k_norm.weight"] = ((hd,), "gain")
            w[p + "mlp.gate_proj.weight"] = w[p + "mlp.up_proj.weight"] = ((F, d), "matrix")
            w[p + "mlp.down_proj.weight"] = ((d, F), "out")
        return w

    def gated(p, d, ff):
        w[p + "gate"] = w[p + "up"] = ((ff, d), "matrix")
        w[p + "down"] = ((d, ff), "out")

    if case["family"] == "miforax":
        z, y = MIFORAX[case["size"]], LATENT
        d, H, r = z["width"], z["heads"], y["kv_rank"]
        w["embed"], w["head"] = ((VOCAB, d), "embedding"), ((VOCAB, d), "matrix")
        w["final.norm"] = ((d,), "gain")
        for i in range(LAYERS):
            p = "l%d.mix." % i
            w["l%d.norm1" % i] = w["l%d.norm2" % i] = ((d,), "gain")
            w[p + "dq"], w[p + "dq.norm"] = ((z["q_rank"], d), "matrix"), ((z["q_rank"],), "gain")
            w[p + "uq"] = ((H * (y["dim"] + y["rot"]), z["q_rank"]), "matrix")
            w[p + "dkv"], w[p + "dkv.norm"] = ((r + y["rot"], d), "matrix"), ((r,), "gain")
            w[p + "uk"], w[p + "uv"] = ((H * y["dim"], r), "matrix"), ((H * y["vdim"], r), "matrix")
            w[p + "sink"] = ((H,), "unit")
            w[p + "g"], w[p + "o"] = ((H * y["vdim"], d), "matrix"), ((d, H * y["vdim"]), "out")
            if i % 2 == 0:
                gated("l%d.mlp." % i, d, z["ff"])
                continue
            w["l%d.mlp.table" % i] = ((VOCAB, z["top"]), "table")
            gated("l%d.mlp.shared." % i, d, z["shared_ff"])
            for e in range(z["experts"]):
                gated("l%d.mlp.e%d." % (i, e), d, z["expert_ff"])
        return w
    z, y = KEBEPEL[case["size"]], WIDE
    d, dk, dv = z["width"], y["dim"], y["vdim"]

    def biased(p, rows):
        w[p], w[p + ".b"] = ((rows, d), "matrix"), ((rows,), "bias")

    def norm(p):
        w[p], w[p + ".b"] = ((d,), "gain"), ((d,), "bias")

    w["embed"], w["head"] = ((VOCAB, d), "embedding"), ((VOCAB, d), "matrix")
    norm("final.norm")
    for i in range(LAYERS):
        for n in ("norm1", "norm1b", "norm2", "norm2b"):
            norm("l%d.%s" % (i, n))
        gated("l%d.mlp." % i, d, z["ff"])
        if i % 2:
            p, H, G, v = "l%d.mix." % i, z["d_heads"], y["d_kv_heads"], y["d_vdim"]
            for n, rows in (("q", H * 2 * dk), ("k", G * 2 * dk), ("v", G * v)):
                biased(p + n, rows)
            for n in ("lq1", "lq2", "lk1", "lk2"):
                w[p + n] = ((dk,), "lambda")
            w[p + "g"], w[p + "o"] = ((H * v, d), "matrix"), ((d, H * v), "out")
            continue
        p, H, G = "l%d.mix.left." % i, z["heads"], z["kv_heads"]
        for n, rows in (("q", H * dk), ("k", G * dk), ("v", G * dv)):
            biased(p + n, rows)
        w[p + "q.norm"], w[p + "k.norm"] = ((H * dk,), "gain"), ((G * dk,), "gain")
        w[p + "g"], w[p + "o"] = ((H * dv, d), "matrix"), ((d, H * dv), "out")
        p, H, G = "l%d.mix.right." % i, z["r_heads"], z["r_kv_heads"]
        for n, rows in (("q", G * dk), ("k", G * dk), ("v", H * dv)):
            w[p + n], w[p + n + ".conv"] = ((rows, d), "matrix"), ((rows, y["conv"]), "taps")
        w[p + "b"] = w[p + "a"] = ((H, d), "matrix")
        w[p + "A_log"], w[p + "dt_bias"], w[p + "norm"] = ((H,), "rate"), ((H,), "step"), ((dv,), "gain")
        w[p + "g"], w[p + "o"] = ((H * dv, d), "matrix"), ((d, H * dv), "out")
    return w


class Weights:
    """The model's tensors by name, each made when it is asked for from the seed and its name: what a reader of a
    checkpoint gives the engine."""

    def __init__(self, case, seed):
        self.table = tensors_of(case)
        self.seed = seed
        self.stored = torch.float32 if case["dtype"] == "fp32" else torch.bfloat16
        self.sublayers = 2 * (QWEN3[case["size"]][0] if case["family"] == "qwen3" else LAYERS)
        self.experts = MIFORAX[case["size"]]["experts"] if case["family"] == "miforax" else 0

    def names(self):
        return list(self.table)

    def shape(self, name):
        return self.table[name][0]

    def dtype(self, name):
        return torch.int32 if self.table[name][1] == "table" else self.stored

    def get(self, name):
        shape, how = self.table[name]
        g = torch.Generator(device="cuda")
        g.manual_seed((int(self.seed) * 1000003 + zlib.crc32(name.encode())) % (2 ** 63 - 1))
        if how == "table":  # every token id names `top` different experts
            return torch.rand((shape[0], self.experts), generator=g, device="cuda").argsort(dim=1)[:, :shape[1]].to(torch.int32).contiguous()
        t = torch.empty(shape, dtype=self.stored if len(shape) == 2 else torch.float32, device="cuda")
        if how == "rate":  # A_log: the logarithm of a rate between 1 and 16
            t.uniform_(0.0, math.log(16.0), generator=g)
        elif how == "step":  # softplus(dt_bias) between 0.001 and 0.1, spread over its logarithm
            t = torch.log(torch.expm1(torch.exp(t.uniform_(math.log(0.001), math.log(0.1), generator=g))))
        else:
            mean, std = {"embedding": (0.0, 0.5), "matrix": (0.0, shape[-1] ** -0.5), "out": (0.0, (shape[-1] * self.sublayers) ** -0.5),
                         "gain": (1.0, 0.1), "bias": (0.0, 0.02), "unit": (0.0, 1.0), "taps": (0.0, 0.5), "lambda": (0.0, 0.1)}[how]
            t.normal_(mean, std, generator=g)
        return t.to(self.stored)


def tokens_of(case, seed):
    """Every request's tokens: its prompt, and behind it the tokens that the pass gives it one by one."""
    vocab = QWEN3_VOCAB if case["family"] == "qwen3" else VOCAB
    more = {"decode": 1, "mixed": 1, "serve": case.get("tokens", 0)}.get(case["kind"], 0)
    sizes = [n + more for n in lengths_of(case)]
    if case["kind"] == "mixed":
        sizes.append(case["behind"] + case["portion"])
    g = torch.Generator()
    g.manual_seed(int(seed) * 7919 + 13)
    return [torch.randint(0, vocab, (n,), generator=g).tolist() for n in sizes]


# ------------------------------------------------------------------------------------------------ what is measured


def prepare(case, seed):
    """The model, its runner (weights, cache, captured steps) and the requests that are already running."""
    tokens, held = tokens_of(case, seed), lengths_of(case)
    model = build_model(parse_config(config_of(case)), Weights(case, seed), "float32" if case["dtype"] == "fp32" else "bfloat16",
                        torch.device("cuda", torch.cuda.current_device()), POSITIONS)
    room = sum(-(-len(t) // PAGE) * PAGE + 4 * PAGE for t in tokens)
    runner = build_runner(model, page_size=PAGE, pool_tokens=room, max_requests=PLACES, max_positions=POSITIONS)
    state = dict(case=case, runner=runner, tokens=tokens, held=held)
    if case["kind"] in ("decode", "mixed"):
        begun = [("r%d" % i, t[:n]) for i, (t, n) in enumerate(zip(tokens, held))]
        if case["kind"] == "mixed" and case["behind"]:
            begun.append(("new", tokens[-1][:case["behind"]]))
        batch, rows = [], 0
        for rid, prompt in begun:  # portions, several requests' together where they are short
            for at in range(0, len(prompt), PORTION):
                part = prompt[at:at + PORTION]
                if rows + len(part) > PORTION or any(e.rid == rid for e in batch):
                    runner.step(batch)
                    batch, rows = [], 0
                batch.append(StepEntry(rid, part))
                rows += len(part)
        runner.step(batch)
    if case["kind"] in ("decode", "serve"):
        run(state)  # the steps of one token are captured once in a program's life
    return state


def run(state):
    case, runner, tokens, held = state["case"], state["runner"], state["tokens"], state["held"]
    if case["kind"] in ("decode", "mixed"):
        entries = [StepEntry("r%d" % i, t[n:n + 1], (0,)) for i, (t, n) in enumerate(zip(tokens, held))]
        if case["kind"] == "mixed":
            entries.append(StepEntry("new", tokens[-1][case["behind"]:], (case["portion"] - 1,)))
        logits = runner.step(entries)
        for e, n in zip(entries, held):
            runner.cache.truncate(e.rid, n)
        if case["kind"] == "mixed":
            if case["behind"]:
                runner.cache.truncate("new", case["behind"])
            else:
                runner.finish("new")
        return logits
    rids = ["r%d" % i for i in range(len(held))]
    logits = [runner.step([StepEntry(rid, t[:n], (n - 1,)) for rid, t, n in zip(rids, tokens, held)])]
    for k in range(case.get("tokens", 0)):  # (a captured step's logits are overwritten by the next one)
        logits.append(runner.step([StepEntry(rid, t[n + k:n + k + 1], (0,)) for rid, t, n in zip(rids, tokens, held)]).clone())
    for rid in rids:
        runner.finish(rid)
    return logits if len(logits) > 1 else logits[0]


# ------------------------------------------------------------------------------------------------ what it takes


def sizes_of(case):
    """Of one layer stack: weights a row passes through, weights a step of n rows reads, cached numbers per position, the
    window, flops per (row, key) pair and per row beside its weights, fp32 numbers of state per request, vocabulary, width."""
    if case["family"] == "qwen3":
        L, d, H, G, hd, F = QWEN3[case["size"]]
        per_row = L * ((2 * H + 2 * G) * hd * d + 3 * d * F)
        return per_row, lambda n: per_row, 2 * L * G * hd, 0, 4 * H * hd * L, 0, 0, QWEN3_VOCAB, d
    if case["family"] == "miforax":
        z, y = MIFORAX[case["size"]], LATENT
        d, H, r = z["width"], z["heads"], y["kv_rank"]
        mixer = (z["q_rank"] + r + y["rot"] + 2 * H * y["vdim"]) * d + H * (y["dim"] + y["rot"]) * z["q_rank"] + H * (y["dim"] + y["vdim"]) * r
        expert, half = 3 * d * z["expert_ff"], LAYERS // 2
        fixed = LAYERS * mixer + half * 3 * d * (z["ff"] + z["shared_ff"])

        def read(n):  # of the experts those that at least one of n rows names
            return fixed + half * expert * z["experts"] * (1.0 - (1.0 - z["top"] / z["experts"]) ** n)
        pair = 2 * H * (y["dim"] + y["rot"] + y["vdim"]) * LAYERS
        return fixed + half * z["top"] * expert, read, LAYERS * (r + y["rot"]), z["window"], pair, 0, 0, VOCAB, d
    z, y = KEBEPEL[case["size"]], WIDE
    d, dk, dv, half = z["width"], y["dim"], y["vdim"], LAYERS // 2
    left = (z["heads"] * (dk + 2 * dv) + z["kv_heads"] * (dk + dv)) * d
    right = (2 * z["r_kv_heads"] * dk + 3 * z["r_heads"] * dv + 2 * z["r_heads"]) * d
    diff = (z["d_heads"] * (2 * dk + 2 * y["d_vdim"]) + y["d_kv_heads"] * (2 * dk + y["d_vdim"])) * d
    per_row = half * (left + right + diff) + LAYERS * 3 * d * z["ff"]
    cached = half * (z["kv_heads"] * (dk + dv) + y["d_kv_heads"] * (2 * dk + y["d_vdim"]))
    pair = half * (2 * z["heads"] * (dk + dv) + 4 * z["d_heads"] * (dk + y["d_vdim"]))
    return per_row, lambda n: per_row, cached, 0, pair, half * 6 * z["r_heads"] * dk * dv, half * z["r_heads"] * dk * dv, VOCAB, d


def steps_of(case):
    """The steps of one pass, each as [(position of the first row, rows)] per request."""
    held = lengths_of(case)
    if case["kind"] == "decode":
        return [[(n, 1) for n in held]]
    if case["kind"] == "mixed":
        return [[(n, 1) for n in held] + [(case["behind"], case["portion"])]]
    return [[(0, n) for n in held]] + [[(n + k, 1) for n in held] for k in range(case.get("tokens", 0))]


def work(case):
    per_row, read, cached, window, pair_flops, row_flops, state, vocab, width = sizes_of(case)
    esize = 4 if case["dtype"] == "fp32" else 2
    by = fl = 0.0
    for step in steps_of(case):
        rows = sum(n for _, n in step)
        keys = sum(min(at, window) if window else at for at, _ in step)
        pairs = sum(sum(min(p + 1, window) for p in range(at, at + n)) if window else n * at + n * (n + 1) / 2 for at, n in step)
        by += (read(rows) + vocab * width + rows * width) * esize + (keys + rows) * cached * esize + len(step) * (vocab + 2 * state) * 4
        fl += rows * (2.0 * per_row + row_flops) + pairs * pair_flops + 2.0 * len(step) * vocab * width
    return {"bytes": by, "flops": fl}


def tolerance(case):
    """Four times what the outputs are off by against float64. bf16: products of rounded inputs through every layer, the last
    one's rounding in front; the heads of the delta rule and of the differential attention are divided by their own root mean
    square, which blows rounding up where they nearly cancel. float32: the order of sums."""
    if case["dtype"] == "fp32":
        return {"rel": 4e-6, "max": 4e-5}
    rel = 0.03 if case["family"] == "kebepel" else 0.01
    return {"rel": rel, "max": 10 * rel}


# ------------------------------------------------------------------------------------------------ the same in 64 bits


def rms(x, gain=None):
    y = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS)
    return y if gain is None else y * gain


def layer_norm(x, gain, bias):
    x = x - x.mean(dim=-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + EPS) * gain + bias


def angles(dims, base, scaling, positions):
    """cos and sin of position * frequency, [rows, 1, dims / 2]; with YaRN where ``scaling`` is given."""
    i = torch.arange(dims // 2, dtype=torch.float64, device="cuda")
    f, amp = base ** (-2.0 * i / dims), 1.0
    if scaling:
        def at(turns):
            return dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
        low, high = max(math.floor(at(scaling["fast"])), 0), min(math.ceil(at(scaling["slow"])), dims - 1)
        ramp = ((i - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
        f, amp = f / scaling["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0
    a = positions.to(torch.float64)[:, None, None] * f
    return torch.cos(a) * amp, torch.sin(a) * amp


def rotated(x, cos, sin, pairs):
    """x [rows, heads, n] with its first entries rotated: halves of the rotated part, or neighbours (``pairs``), belong together."""
    n = 2 * cos.shape[-1]
    u, v = (x[..., 0:n:2], x[..., 1:n:2]) if pairs else (x[..., :n // 2], x[..., n // 2:n])
    a, b = u * cos - v * sin, v * cos + u * sin
    front = torch.stack([a, b], dim=-1).flatten(-2) if pairs else torch.cat([a, b], dim=-1)
    return torch.cat([front, x[..., n:]], dim=-1)


def attend(q, k, v, scale, window=0, sink=None, cap=0.0):
    """Causal softmax attention of one sequence: q [T, H, d], k [T, G, d], v [T, Gv, dv] -> [T, H, dv]."""
    T, H, _ = q.shape
    kt = k.permute(1, 2, 0).repeat_interleave(H // k.shape[1], dim=0).contiguous()
    vh = v.permute(1, 0, 2).repeat_interleave(H // v.shape[1], dim=0).contiguous()
    out = torch.empty(T, H, v.shape[-1], dtype=q.dtype, device=q.device)
    step = max(16, min(T, (1 << 28) // (H * T)))
    for a in range(0, T, step):
        b = min(T, a + step)
        s = torch.matmul(q[a:b].transpose(0, 1).contiguous(), kt[:, :, :b].contiguous()) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        i, j = torch.arange(a, b, device=q.device)[:, None], torch.arange(b, device=q.device)[None]
        s = s.masked_fill((j > i) | ((i - j >= window) if window else (j > i)), float("-inf"))
        top = s.amax(dim=-1, keepdim=True)
        if sink is not None:
            top = torch.maximum(top, sink[:, None, None])
        e = torch.exp(s - top)
        below = e.sum(dim=-1, keepdim=True) + (torch.exp(sink[:, None, None] - top) if sink is not None else 0.0)
        out[a:b] = torch.matmul(e / below, vh[:, :b].contiguous()).transpose(0, 1)
    return out


def per_sequence(f, parts, *tensors):
    return torch.cat([f(*(t[a:b] for t in tensors)) for a, b in parts])


def qwen3_rows(case, get, ids, positions, parts, last):
    L, d, H, G, hd, F = QWEN3[case["size"]]
    cos, sin = angles(hd, QWEN3_BASE, None, positions)
    x = get("model.embed_tokens.weight", ids)
    for i in range(L):
        p = "model.layers.%d." % i
        h = rms(x, get(p + "input_layernorm.weight"))
        q, k, v = (h @ get(p + "self_attn.%s_proj.weight" % n).t() for n in "qkv")
        q, k = rms(q.view(-1, H, hd), get(p + "self_attn.q_norm.weight")), rms(k.view(-1, G, hd), get(p + "self_attn.k_norm.weight"))
        q, k = rotated(q, cos, sin, False), rotated(k, cos, sin, False)
        a = per_sequence(lambda q, k, v: attend(q, k, v, hd ** -0.5), parts, q, k, v.view(-1, G, hd))
        x = x + a.reshape(-1, H * hd) @ get(p + "self_attn.o_proj.weight").t()
        h = rms(x, get(p + "post_attention_layernorm.weight"))
        g = h @ get(p + "mlp.gate_proj.weight").t()
        g = torch.nn.functional.silu(g).mul_(h @ get(p + "mlp.up_proj.weight").t())
        x = x + g @ get(p + "mlp.down_proj.weight").t()
    return rms(x[last], get("model.norm.weight")) @ get("lm_head.weight").t()


def miforax_rows(case, get, ids, positions, parts, last):
    z, y = MIFORAX[case["size"]], LATENT
    H, r = z["heads"], y["kv_rank"]
    scale = (y["dim"] + y["rot"]) ** -0.5
    cos, sin = angles(y["rot"], 1e6, YARN, positions)

    def expert(h, p):
        g, u = (h @ get(p + "gate").t()).clamp(max=7.0), (h @ get(p + "up").t()).clamp(-7.0, 7.0)
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ get(p + "down").t()

    x = get("embed", ids)
    for i in range(LAYERS):
        p = "l%d.mix." % i
        h = rms(x, get("l%d.norm1" % i))
        q = (rms(h @ get(p + "dq").t(), get(p + "dq.norm")) @ get(p + "uq").t()).view(-1, H, y["dim"] + y["rot"])
        q = torch.cat([q[..., :y["dim"]], rotated(q[..., y["dim"]:], cos, sin, False)], dim=-1)
        ckr = h @ get(p + "dkv").t()
        c = rms(ckr[:, :r], get(p + "dkv.norm"))
        k = torch.cat([(c @ get(p + "uk").t()).view(-1, H, y["dim"]), rotated(ckr[:, None, r:], cos, sin, False).expand(-1, H, -1)], dim=-1)
        v, sink = (c @ get(p + "uv").t()).view(-1, H, y["vdim"]), get(p + "sink")
        a = per_sequence(lambda q, k, v: attend(q, k, v, scale, z["window"], sink), parts, q, k, v)
        x = x + (a.reshape(-1, H * y["vdim"]) * torch.sigmoid(h @ get(p + "g").t())) @ get(p + "o").t()
        h, p = rms(x, get("l%d.norm2" % i)), "l%d.mlp." % i
        if i % 2 == 0:
            x = x + (torch.nn.functional.gelu(h @ get(p + "gate").t(), approximate="tanh") * (h @ get(p + "up").t())) @ get(p + "down").t()
            continue
        more, named = expert(h, p + "shared."), get(p + "table", ids).long()
        for e in range(z["experts"]):
            rows = (named == e).any(dim=1).nonzero()[:, 0]
            more[rows] += expert(h[rows], p + "e%d." % e) / z["top"]
        x = x + more
    return rms(x[last], get("final.norm")) @ get("head").t()


def kebepel_rows(case, get, ids, positions, parts, last):
    z, y = KEBEPEL[case["size"]], WIDE
    dk, dv = y["dim"], y["vdim"]
    scale = dk ** -0.5
    cos, sin = angles(dk, 1e6, YARN, positions)

    def convolved(x, taps):
        def one(x):
            n = taps.shape[1]
            padded = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
            return sum(padded[j:j + x.shape[0]] * taps[:, j] for j in range(n))
        return torch.nn.functional.silu(per_sequence(one, parts, x))

    def unit(x):
        return x / torch.sqrt((x * x).sum(dim=-1, keepdim=True) + 1e-6)

    def delta(q, k, v, beta, decay):
        S = q.new_zeros(q.shape[1], dk, dv)
        out = []
        for t in range(q.shape[0]):
            S = S * decay[t][:, None, None]
            S = S + k[t][:, :, None] * (beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(dim=1)))[:, None]
            out.append((S * q[t][:, :, None]).sum(dim=1))
        return torch.stack(out)

    def left(h, p):
        H, G = z["heads"], z["kv_heads"]
        q, k, v = (h @ get(p + n).t() + get(p + n + ".b") for n in "qkv")
        q, k = (rotated(rms(t, get(p + n + ".norm")).view(-1, c, dk), cos, sin, True) for t, n, c in ((q, "q", H), (k, "k", G)))
        a = per_sequence(lambda q, k, v: attend(q, k, v, scale, cap=30.0), parts, q, k, v.view(-1, G, dv))
        return (a.reshape(-1, H * dv) * torch.sigmoid(h @ get(p + "g").t())) @ get(p + "o").t()

    def right(h, p):
        H, G = z["r_heads"], z["r_kv_heads"]
        q, k, v = (convolved(h @ get(p + n).t(), get(p + n + ".conv")) for n in "qkv")
        q = (unit(q.view(-1, G, dk)) * scale).repeat_interleave(H // G, dim=1)
        k = unit(k.view(-1, G, dk)).repeat_interleave(H // G, dim=1)
        beta = torch.sigmoid(h @ get(p + "b").t())
        decay = torch.exp(-torch.exp(get(p + "A_log")) * torch.nn.functional.softplus(h @ get(p + "a").t() + get(p + "dt_bias"), threshold=50.0))
        o = rms(per_sequence(delta, parts, q, k, v.view(-1, H, dv), beta, decay), get(p + "norm"))
        return (o.reshape(-1, H * dv) * torch.nn.functional.silu(h @ get(p + "g").t())) @ get(p + "o").t()

    def differential(h, p):
        H, G, n = z["d_heads"], y["d_kv_heads"], y["d_vdim"]
        q, k, v = (h @ get(p + c).t() + get(p + c + ".b") for c in "qkv")
        q = q.view(-1, H, 2, dk) * (1.0 + 0.1 * torch.log(torch.floor((positions.to(torch.float64) + 1.0) / 256) + 1.0))[:, None, None, None]
        k, v = k.view(-1, G, 2, dk), v.view(-1, G, n)
        a, b = (per_sequence(lambda q, k, v: attend(q, k, v, scale), parts, q[:, :, m], k[:, :, m], v) for m in (0, 1))
        lam = torch.exp((get(p + "lq1") * get(p + "lk1")).sum()) - torch.exp((get(p + "lq2") * get(p + "lk2")).sum()) + 0.2
        o = rms(a - lam * b) * 0.8
        return (o.reshape(-1, H * n) * torch.sigmoid(h @ get(p + "g").t())) @ get(p + "o").t()

    def norm(x, n):
        return layer_norm(x, get(n), get(n + ".b"))

    x = get("embed", ids)
    for i in range(LAYERS):
        h, p = norm(x, "l%d.norm1" % i), "l%d.mix." % i
        x = x + norm(differential(h, p) if i % 2 else left(h, p + "left.") + right(h, p + "right."), "l%d.norm1b" % i)
        h, p = norm(x, "l%d.norm2" % i), "l%d.mlp." % i
        x = x + norm((torch.nn.functional.silu(h @ get(p + "gate").t()) * (h @ get(p + "up").t())) @ get(p + "down").t(), "l%d.norm2b" % i)
    return norm(x[last], "final.norm") @ get("head").t()


def exact(case, seed):
    """The logits of ``run`` in float64: whole sequences, no cache."""
    tokens, source = tokens_of(case, seed), Weights(case, seed)
    if sum(len(t) for t in tokens) * 2.0 * sizes_of(case)[0] > 5e14:
        return None

    def get(name, rows=None):
        t = source.get(name)
        return (t if rows is None else t[rows]).to(torch.float64)

    parts, at = [], 0
    for t in tokens:
        parts.append((at, at + len(t)))
        at += len(t)
    ids = torch.tensor([i for t in tokens for i in t], device="cuda")
    positions = torch.cat([torch.arange(len(t), device="cuda") for t in tokens])
    steps = 1 + (case.get("tokens", 0) if case["kind"] == "serve" else 0)  # a request's wanted rows are its last ones
    last = torch.tensor([b - steps + k for k in range(steps) for _, b in parts], device="cuda")
    rows = {"qwen3": qwen3_rows, "miforax": miforax_rows, "kebepel": kebepel_rows}[case["family"]](case, get, ids, positions, parts, last)
    rows = list(rows.view(steps, len(parts), -1))
    return rows if steps > 1 else rows[0]
