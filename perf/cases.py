"""What this engine is measured by: steps of served models, as a server, a batch job or an evaluation runs them.

A pass is one step through ``ModelRunner.step``, the step function under ``Engine`` and the trace replay: token ids in, float32
logits at the wanted places out.  Three kinds of steps:

* ``decode``: every live request brings one token (the captured step that ``Engine`` replays for each new token);
* ``prefill``: prompts arrive, run whole in one step, and give their pages back (the first token of a request, or scoring);
* ``mixed``: a portion of a prompt beside decoding requests (continuous batching under a token budget).

The models are those of ``bench.py``: the Llama 3 decoder at its 1B and 8B shapes, in bfloat16 and in the true 32-bit path, and
the other designs at the 1B shape with bench.py's head counts, experts and ranks.  Weights are random by the laws that the
parts name (linear N(0, 0.02), norms 1 + N(0, 0.02), decays and convolutions by their own), with embeddings N(0, 1) and
smaller writes into the stream (``BEHIND``), drawn on the GPU from the seed.
Depths are cut (8 of the 8B shape's 32 layers, 4 to 8 of the designs' 16; ``bench.py --layers`` does the same) so that a model
is made in about a second; every weight matrix keeps its size, and the weights are far more than any cache holds.  Prompts
are uniform random token ids.  Lengths within a step are ragged, as those of a server's requests are.

The Fetitar design is left out: its mixers run on the kernels of those here (attention through a latent, attention with
keys and values of two sizes) and its feed-forwards on Llama's.
"""

from __future__ import annotations

import math
import zlib

import torch

DEV = "cuda"
PAGE = 16
GROWTH = 3072  # tokens that the decoding requests of a state may grow by before they start anew

LLAMA = {
    "1b": dict(hidden_size=2048, intermediate_size=8192, num_hidden_layers=16, num_attention_heads=32, num_key_value_heads=8, head_dim=64,
               tie_word_embeddings=True, factor=32.0),
    "8b": dict(hidden_size=4096, intermediate_size=14336, num_hidden_layers=32, num_attention_heads=32, num_key_value_heads=8, head_dim=128,
               tie_word_embeddings=False, factor=8.0),
}
VOCAB = 128256
DESIGNS = ("vuzelix", "padetar", "fimilorn", "zipedra", "meropel")


def listed():
    return [
        # one user, a chat at a context of about a thousand tokens: the latency of a token, 100 kernels that each read a few megabytes
        dict(name="llama1b-decode-1", model="llama", shape="1b", layers=16, dtype="bf16", kind="decode", requests=1, context=1100, tokens=0),
        # the benchmark's decode: eight requests at a context of about 3,072
        dict(name="llama8b-decode-8", model="llama", shape="8b", layers=8, dtype="bf16", kind="decode", requests=8, context=3072, tokens=0),
        # a loaded server: 61 requests (a captured step of 64 rows), the cache a large part of what is read
        dict(name="llama8b-decode-61", model="llama", shape="8b", layers=8, dtype="bf16", kind="decode", requests=61, context=2100, tokens=0),
        # the benchmark's prompt of 2,048 tokens
        dict(name="llama8b-prefill-2048", model="llama", shape="8b", layers=8, dtype="bf16", kind="prefill", requests=1, context=0, tokens=2048),
        # serving: a portion of 480 prompt tokens beside 32 decoding requests, a budget of 512
        dict(name="llama1b-mixed-32-480", model="llama", shape="1b", layers=16, dtype="bf16", kind="mixed", requests=32, context=600, tokens=480),
        # the 32-bit path, as an evaluation or a check of a checkpoint uses it: a prompt of odd length
        dict(name="llama1b-fp32-prefill-777", model="llama", shape="1b", layers=8, dtype="fp32", kind="prefill", requests=1, context=0, tokens=777),
        # the 32-bit path generating for a few requests
        dict(name="llama1b-fp32-decode-5", model="llama", shape="1b", layers=8, dtype="fp32", kind="decode", requests=5, context=900, tokens=0),
        # delta-rule layers and attention in chunks: a prompt of the benchmark's length
        dict(name="vuzelix-prefill-2048", model="vuzelix", shape="1b", layers=8, dtype="bf16", kind="prefill", requests=1, context=0, tokens=2048),
        # matrix memory beside attention, experts: three prompts of different lengths in one step
        dict(name="padetar-prefill-3x", model="padetar", shape="1b", layers=4, dtype="bf16", kind="prefill", requests=3, context=0, tokens=1531),
        # latent attention, retention, grouped experts, looped layers: eight requests decoding
        dict(name="fimilorn-decode-8", model="fimilorn", shape="1b", layers=4, dtype="bf16", kind="decode", requests=8, context=2048, tokens=0),
        # latent attention over every earlier position, lightning attention, ungated experts: the benchmark's prompt
        dict(name="zipedra-prefill-2048", model="zipedra", shape="1b", layers=4, dtype="bf16", kind="prefill", requests=1, context=0, tokens=2048),
        # selective scan, gated linear attention, Mamba-2, experts: a portion of 500 tokens beside eight decoding requests
        dict(name="meropel-mixed-8-500", model="meropel", shape="1b", layers=6, dtype="bf16", kind="mixed", requests=8, context=700, tokens=500),
    ]


def draw(rng):
    """Any model, any kind of step, sizes over their logarithm: 1 to 64 requests, contexts of 60 to 4,000, prompts of 17 to 2,048 tokens."""
    log = lambda low, high: int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    model = rng.choice(("llama", "llama", "llama") + DESIGNS)
    shape = rng.choice(("1b", "8b")) if model == "llama" else "1b"
    dtype = "fp32" if model == "llama" and shape == "1b" and rng.random() < 0.3 else "bf16"
    layers = {"llama": 8, "vuzelix": 8, "padetar": 4, "fimilorn": 4, "zipedra": 4, "meropel": 6}[model]
    kind = rng.choice(("decode", "prefill", "prefill", "mixed"))
    case = dict(model=model, shape=shape, layers=layers, dtype=dtype, kind=kind, requests=1, context=0, tokens=0)
    if kind == "decode":
        case["requests"] = log(1, 64) if dtype == "bf16" else log(1, 8)
        case["context"] = log(60, min(4000, 130000 // case["requests"]))
    elif kind == "prefill":
        case["requests"] = rng.choice((1, 1, 2, 3))
        case["tokens"] = log(17 * case["requests"], 2048 if dtype == "bf16" else 777)
    else:
        case["requests"] = log(1, 48) if dtype == "bf16" else log(1, 8)
        case["context"] = log(60, 1500)
        case["tokens"] = log(17, 960 if dtype == "bf16" else 500)
    return case


# ------------------------------------------------------------------ configurations and weights


def _llama_raw(case):
    s = dict(LLAMA[case["shape"]])
    factor = s.pop("factor")
    return dict(s, model_type="llama", vocab_size=VOCAB, num_hidden_layers=case["layers"], rms_norm_eps=1e-5, rope_theta=500000.0,
                max_position_embeddings=131072,
                rope_scaling=dict(rope_type="llama3", factor=factor, low_freq_factor=1.0, high_freq_factor=4.0, original_max_position_embeddings=8192))


def _design_raw(case):
    """The design's config.json with bench.py's sizes for the shape."""
    s = LLAMA[case["shape"]]
    H, G, D, F, W, n = (s["num_attention_heads"], s["num_key_value_heads"], s["head_dim"], s["intermediate_size"], s["hidden_size"], case["layers"])
    design = case["model"]
    raw = {"architecture": design.capitalize(), "vocab": VOCAB, "width": W, "norm": {"eps": 1e-5 if design in ("vuzelix", "padetar") else 1e-6}}
    if design == "vuzelix":
        layers, last = [], None
        for i in range(n):
            mlp = {"kind": "dense", "ff": F}
            if i % 4 == 0:
                layers.append({"type": "channel_delta", "mixer": dict(heads=16, kv_heads=16, dim=128, vdim=128, conv=4), "mlp": mlp})
                continue
            m = dict(heads=H, kv_heads=G, dim=D, vdim=D, scale=D**-0.5, softcap=50.0, mask={"size": 1024})
            if i % 4 == 3:
                m["kv_from"] = last
            last = i if "kv_from" not in m else last
            layers.append({"type": "attention", "mixer": m, "mlp": mlp})
        return dict(raw, layers=layers, embedding={"scale": 1.0}, residual_mult=0.5, streams=4, logit_softcap=30.0)
    if design == "padetar":
        left = dict(heads=H, kv_heads=G, dim=D, vdim=D, scale=D**-0.5,
                    rot={"base": 1e6, "dims": D, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})
        mlp = {"kind": "moe", "router": {"experts": 32, "top": 4}, "expert": {"ff": F // 8, "limit": 7.0}, "shared": {"ff": F // 2, "limit": 7.0}}
        mixer = {"left": left, "left_scale": 1.0, "right": dict(heads=W // 256, dim=128, vdim=256, gate_cap=15.0), "right_scale": 1.0}
        return dict(raw, token_side={"dim": 256}, layers=[{"type": "parallel", "mixer": mixer, "mlp": mlp}] * n)
    latent = dict(heads=H, dim=D, rot_dim=D // 2, vdim=D, kv_rank=512, scale=(D + D // 2) ** -0.5, rot={"base": 1e6, "dims": D // 2})
    decays = [1.0 - 2.0 ** (-5 - h % 8) for h in range(W // 256)]
    if design == "fimilorn":
        mixers = [("attention", dict(heads=H, kv_heads=G, dim=D, vdim=D, scale=D**-0.5, rot={"base": 1e6, "dims": D})),
                  ("latent_attention", dict(latent, mask={"size": 1024})),
                  ("retention", dict(heads=W // 256, dim=128, vdim=256, decay=decays, rot={"base": 1e4, "dims": 128}))]
        moe = {"kind": "moe", "expert": {"ff": F // 8}, "router": {"experts": 32, "top": 4, "groups": {"count": 8, "keep": 4}}, "shared": {"ff": F // 2}}
        layers = [{"type": mixers[i % 3][0], "mixer": mixers[i % 3][1], "mlp": {"kind": "dense", "ff": F, "limit": 7.0} if i == 0 else moe} for i in range(n)]
        return dict(raw, loop={"start": 1, "stop": 4, "times": 2}, layers=layers)
    if design == "zipedra":
        mixers = [("latent_attention", latent), ("lightning", dict(heads=W // 256, dim=128, vdim=256, decay=decays))]
        moe = {"kind": "moe", "expert": {"ff": 3 * F // 16}, "router": {"experts": 32, "top": 4}, "shared": {"ff": 3 * F // 4}}
        layers = [{"type": mixers[i % 2][0], "mixer": mixers[i % 2][1], "mlp": {"kind": "dense", "ff": F} if i == 0 else moe} for i in range(n)]
        return dict(raw, logit_scale=0.5, token_side={"dim": 256}, loop={"start": 1, "stop": 4, "times": 2}, layers=layers)
    half = dict(heads=H // 2, kv_heads=G // 2, dim=D, vdim=2 * D, scale=D**-0.5, rot={"base": 1e6, "dims": D // 2})
    whole = dict(heads=H, kv_heads=G, dim=D, vdim=D, scale=D**-0.5, rot={"base": 1e6, "dims": D})
    mixers = [("parallel", {"left": half, "right": dict(inner=W, state=16, dt_rank=W // 16, conv=4), "left_scale": 1.0, "right_scale": 1.0}),
              ("gla", dict(heads=W // 256, dim=128, vdim=256, tau=16.0)),
              ("parallel_2", {"left": whole, "right": dict(heads=W // 64, vdim=64, state=128, groups=1, conv=4, norm_groups=1)})]
    moe = {"kind": "moe", "expert": {"ff": F // 8}, "shared": {"ff": F // 2},
           "router": {"experts": 32, "top": 4, "scale": 1.5, "identity": 4, "groups": {"count": 4, "keep": 2}}}
    layers = [{"type": mixers[i % 3][0], "mixer": mixers[i % 3][1], "mlp": {"kind": "dense", "ff": F} if i == 0 else moe} for i in range(n)]
    return dict(raw, logit_scale=0.5, embedding={"bigram": {"buckets": 65536, "mul_prev": 127, "mul_cur": 7}}, layers=layers)


def _config(case):
    from nanospec_amd import LlamaConfig
    from nanospec_amd import config as configs

    if case["model"] == "llama":
        return LlamaConfig.from_hf(_llama_raw(case))
    return getattr(configs, case["model"].capitalize() + "Config").from_hf(_design_raw(case))


def _tied(case):
    return case["model"] == "fimilorn" or case["model"] == "llama" and LLAMA[case["shape"]]["tie_word_embeddings"]


RANKS = {"vuzelix": 64, "meropel": 16}  # inner sizes that a checkpoint's tensors tell and config.json does not


# Norms that stand behind a sublayer.  Their weights, and where there are none the matrices that write into the stream, are
# such that a sublayer adds a fraction of the stream's size, as in trained models: a stream that every sublayer turns over
# multiplies each rounding from layer to layer until no two orders of summation agree.
BEHIND = {"padetar": ("norm1", "norm2"), "fimilorn": ("norm1b", "norm2b"), "meropel": ("norm1b", "norm2b")}


def _tensor(case, seed, name, shape):
    """One weight, from the seed and its name alone, in the case's data type."""
    g = torch.Generator(device=DEV)
    g.manual_seed(zlib.crc32(name.encode()) * 1000003 + int(seed))
    t = torch.empty(shape, dtype=torch.float32, device=DEV)
    last = name.rsplit(".", 1)[-1]
    if last == "D":
        t.fill_(1.0)
    elif last == "A_log" and case["model"] == "vuzelix":
        t.uniform_(0.02, 1.0, generator=g).log_()
    elif last == "A_log" and len(shape) == 2:
        t.normal_(0.0, 0.1, generator=g).add_(torch.arange(1, shape[1] + 1, device=DEV).float().log())
    elif last == "A_log":
        t.uniform_(1.0, 16.0, generator=g).log_()
    elif last == "conv":
        t.normal_(0.0, 0.5, generator=g)
    elif name.endswith("right.dt_bias") or name.endswith("dt.b"):
        t.uniform_(-4.6, -1.2, generator=g)
    elif last == "dt_bias":
        t.normal_(0.0, 1.0, generator=g)
    elif name.endswith("a2.b"):
        t.uniform_(-2.0, 3.0, generator=g)
    elif last in ("a2", "g2") and case["model"] == "vuzelix":
        t.normal_(0.0, 0.3, generator=g)
    elif name.endswith("right.f.b"):
        t.uniform_(1.0, 4.0, generator=g)
    elif name.endswith("right.i.b"):
        t.normal_(0.0, 0.5, generator=g)
    elif ".hc" in name and last == "mix":
        t.normal_(0.0, 0.05, generator=g).add_(torch.eye(shape[0], device=DEV) * 0.9 + 0.1 / shape[0])
    elif ".hc" in name:
        t.normal_(0.0, 0.1, generator=g).add_(1.0 / 4 if last == "in" else 1.0)
    elif last == "sink":
        t.normal_(0.0, 0.1, generator=g)
    elif last in BEHIND.get(case["model"], ()):
        t.normal_(0.125, 0.02, generator=g)
    elif last in ("embed", "weight") and "embed" in name and not name.startswith("side"):
        t.normal_(0.0, 1.0, generator=g)
    elif "norm" in name or name.endswith("left.out") or name.endswith("right.out"):
        t.normal_(1.0, 0.02, generator=g)
    elif case["model"] not in BEHIND and (last in ("o", "down") or "o_proj" in name or "down_proj" in name):
        t.normal_(0.0, 0.005, generator=g)
    else:
        t.normal_(0.0, 0.02, generator=g)
    return t.to(torch.bfloat16 if case["dtype"] == "bf16" else torch.float32)


class _Weights:
    """A checkpoint as ``DecoderModel.load`` reads one: names, shapes, tensors."""

    where = "<seeded random>"

    def __init__(self, case, seed, wanted):
        self.case, self.seed = case, seed
        rank = RANKS.get(case["model"])
        self._shapes = {k: tuple(rank if d is None else d for d in shape) for k, (shape, _) in wanted.items()}
        if _tied(case):  # the embedding table is the head
            self._shapes.pop("lm_head.weight" if case["model"] == "llama" else "head")

    def names(self):
        return list(self._shapes)

    def shape(self, name):
        return self._shapes[name]

    def get(self, name):
        return _tensor(self.case, self.seed, name, self._shapes[name])


# ------------------------------------------------------------------ requests


def _contexts(case):
    """Tokens that each decoding request has in the cache before the pass: within a quarter of the context, all different."""
    c = case["context"]
    return [max(1, c - (37 * i) % (c // 4 + 1)) for i in range(case["requests"])] if case["kind"] != "prefill" else []


def _prompts(case):
    """Lengths of the prompts that a pass brings."""
    if case["kind"] == "decode":
        return []
    n = case["requests"] if case["kind"] == "prefill" else 1
    total = case["tokens"]
    lens = [max(1, total * (i + 1) // (n * (n + 1) // 2)) for i in range(n - 1)]
    return lens + [total - sum(lens)]


def _ids(case, seed, request, n):
    g = torch.Generator()
    g.manual_seed(int(seed) * 1009 + request)
    return torch.randint(0, VOCAB, (n,), generator=g).tolist()


LEAD = 2  # tokens that the decoding requests have decoded before the first pass (the step's shape is captured by then)


def prepare(case, seed):
    """A loaded model, a cache with the decoding requests in it, and the prompts that arrive."""
    from nanospec_amd.engine.replay import Replayer
    from nanospec_amd.parts import DecoderModel

    cfg = _config(case)
    model = DecoderModel(cfg.model_spec(), cfg)
    model.load(_Weights(case, seed, model.wanted()), torch.bfloat16 if case["dtype"] == "bf16" else torch.float32, torch.device(DEV))
    contexts, prompts = _contexts(case), _prompts(case)
    room = sum(-(-(c + GROWTH + LEAD) // PAGE) + 1 for c in contexts) if case["kind"] != "prefill" else 0
    room += sum(-(-p // PAGE) + 1 for p in prompts)
    # (a decoding request may grow by GROWTH tokens in all; the requests of a step share the pool)
    rep = Replayer(model, PAGE * room, page_size=PAGE, max_live=len(contexts) + len(prompts))
    state = {"runner": rep.runner, "manager": rep.manager, "prompts": [(f"p{i}", _ids(case, seed, 1000 + i, n)) for i, n in enumerate(prompts)],
             "requests": [(f"d{i}", _ids(case, seed, i, c + LEAD + GROWTH)) for i, c in enumerate(contexts)], "contexts": contexts}
    _start(state)
    if case["kind"] == "prefill" and case["tokens"] <= 1024 or case["kind"] == "mixed":
        run(state)  # the step's shape is captured
        _restart(state)
    return state


def _start(state):
    """The decoding requests' prompts, some at a time, and their first decoded tokens."""
    from nanospec_amd.engine.runner import StepEntry

    runner = state["runner"]
    with torch.cuda.stream(runner.stream):
        for (rid, ids), c in zip(state["requests"], state["contexts"]):
            runner.admit(rid)
            for at in range(0, c, 2048):
                runner.step([StepEntry(rid, ids[at : min(c, at + 2048)], [])])
        for k in range(LEAD if state["requests"] else 0):
            runner.step([StepEntry(rid, [ids[c + k]], [0]) for (rid, ids), c in zip(state["requests"], state["contexts"])])
    runner.synchronize()


def _restart(state):
    for rid, _ in state["requests"]:
        state["runner"].release(rid)
    _start(state)


def run(state):
    """One step: the next token of every decoding request and the prompts that arrive; -> its logits.  A prompt's pages
    go back after it (its request is done or, beside decoding ones, is preempted), so the next pass finds the same cache
    but for the tokens that the decoding requests have gained."""
    from nanospec_amd.engine.runner import StepEntry

    runner, manager = state["runner"], state["manager"]
    if state["requests"] and manager.get(state["requests"][0][0]).length >= len(state["requests"][0][1]):
        _restart(state)  # the requests have reached their longest: others take their places
    entries = [StepEntry(rid, [ids[manager.get(rid).length]], [0]) for rid, ids in state["requests"]]
    with torch.cuda.stream(runner.stream):  # as Engine.step
        for rid, ids in state["prompts"]:
            runner.admit(rid)
            entries.append(StepEntry(rid, ids, [len(ids) - 1]))
        logits = runner.step(entries)
        for rid, _ in state["prompts"]:
            runner.release(rid)
    return logits


# ------------------------------------------------------------------ what a pass cannot do without


def _mixers(case):
    """(kind, sizes) of every mixer that runs, a looped layer once a pass."""
    if case["model"] == "llama":
        s = LLAMA[case["shape"]]
        return [("attention", dict(heads=s["num_attention_heads"], kv_heads=s["num_key_value_heads"], dim=s["head_dim"], vdim=s["head_dim"]))] * case["layers"]
    raw, out = _design_raw(case), []
    for i in _order(raw):
        e = raw["layers"][i[0]]
        m = e["mixer"]
        if e["type"] == "parallel" or e["type"] == "parallel_2":
            right = m["right"]
            state = ({"heads": right["inner"], "dim": right["state"], "vdim": 1} if "inner" in right
                     else {"heads": right["heads"], "dim": right.get("state", right.get("dim")), "vdim": right["vdim"]})
            out += [("attention", m["left"]), ("recurrence", state)]
        elif e["type"] in ("attention", "latent_attention"):
            out.append((e["type"], m))
        else:
            out.append(("recurrence", m))
    return out


def _order(raw):
    """(layer, number of the pass that starts in front of it or None) in the order the layers run."""
    n, loop = len(raw["layers"]), raw.get("loop")
    if not loop:
        return [(i, None) for i in range(n)]
    a, b = loop["start"], loop["stop"]
    inside = [(i, t if i == a else None) for t in range(loop["times"]) for i in range(a, b)]
    return [(i, None) for i in range(a)] + inside + [(i, None) for i in range(b, n)]


def _pairs(first, n, mixer):
    """(query, key) pairs of ``n`` new tokens behind ``first`` cached ones."""
    size = (mixer.get("mask") or {}).get("size", 1 << 40)
    return sum(min(first + i + 1, size) for i in range(n))


def work(case):
    from nanospec_amd.parts.model import wanted_tensors

    size = 2 if case["dtype"] == "bf16" else 4
    portions = [(c + LEAD, 1) for c in _contexts(case)] + [(0, n) for n in _prompts(case)]
    tokens, rows = sum(n for _, n in portions), len(portions)
    times = {}
    if case["model"] != "llama":
        for i, _ in _order(_design_raw(case)):
            times[f"l{i}"] = times.get(f"l{i}", 0) + 1
    read, flops = 0.0, 0.0
    for name, (shape, _) in wanted_tensors(_config(case).model_spec()).items():
        n = math.prod(RANKS.get(case["model"]) if d is None else d for d in shape)
        passes = times.get(name.split(".")[0], 1)
        if "embed" in name or name == "bigram":
            read += tokens * shape[1] * size
        elif ".mlp.e" in name:  # 32 experts, four a token
            read += n * size * (1 - (1 - 4 / 32) ** (tokens * passes))
            flops += 2.0 * n * tokens * passes * 4 / 32
        else:
            read += n * size
            flops += 2.0 * n * (rows if name in ("lm_head.weight", "head") else tokens * passes) if len(shape) == 2 else 0.0
    for kind, m in _mixers(case):
        if kind == "recurrence":
            read += 2.0 * rows * m["heads"] * m["dim"] * m["vdim"] * 4
            flops += 4.0 * tokens * m["heads"] * m["dim"] * m["vdim"]
            continue
        per_key = m["kv_rank"] + m["rot_dim"] if kind == "latent_attention" else m["kv_heads"] * (m["dim"] + m["vdim"])
        window = (m.get("mask") or {}).get("size", 1 << 40)
        read += size * per_key * (sum(min(first, window) for first, _ in portions) + tokens)
        flops += 2.0 * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m["vdim"]) * sum(_pairs(first, n, m) for first, n in portions)
    return {"bytes": read + rows * VOCAB * 4.0, "flops": flops}


def tolerance(case):
    """bfloat16: the outputs of every product and part are rounded to 8 bits, and a sum in another order changes some of them by
    a unit in the last place.  The same requests through other kernels of the start (rows alone instead of in a batch, prompts
    in two portions, norms as kernels of their own) differ by 0.3 to 1.2% in the 2-norm, 0.07 of the root mean square at most, and
    by 1.7% and 0.18 where a token's router scores lie within rounding of each other and it takes another expert.  32-bit: 1.2e-6
    from 64 bits."""
    return {"rel": 1e-5, "max": 2e-4} if case["dtype"] == "fp32" else {"rel": 0.03, "max": 0.5}


# ------------------------------------------------------------------ the same in 64 bits


def exact(case, seed):
    """The logits of the first pass from plain whole-sequence arithmetic in 64 bits, from the designs' equations."""
    new = [(c + LEAD + 1, i) for i, c in enumerate(_contexts(case))] + [(n, 1000 + i) for i, n in enumerate(_prompts(case))]
    steps = sum(n for n, _ in new) * len(_mixers(case)) * (0.0 if case["model"] == "llama" else 6e-5)  # recurrences, a token at a time
    params = 0.9e9 if case["shape"] == "1b" else 0.22e9 * case["layers"]
    if steps + 2 * params * sum(n for n, _ in new) / 2e13 > 18:
        return None
    plain = _Plain(case, seed)
    length = {i: c + LEAD + GROWTH for i, c in enumerate(_contexts(case))}
    return torch.cat([plain.logits(_ids(case, seed, r, length.get(r, n))[:n]) for n, r in new])


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z**3)))


def _softplus(z):
    return z.clamp(min=0) + torch.log1p(torch.exp(-z.abs()))


def _frequencies(dims, base, scaling=None):
    """base^(-2 i / dims); long wavelengths ``factor`` times slower, a linear blend between the two borders."""
    out = []
    for i in range(dims // 2):
        f = base ** (-2.0 * i / dims)
        if scaling:
            factor, low, high, span = scaling
            wave = 2 * math.pi / f
            if wave > span / low:
                f /= factor
            elif wave >= span / high:
                s = (span / wave - low) / (high - low)
                f = (1 - s) * f / factor + s * f
        out.append(f)
    return torch.tensor(out, dtype=torch.float64, device=DEV)


def _rotate(x, freq, interleaved=False):
    """x [T, heads, >= 2 len(freq)]: pairs (i, i + half), or (2 i, 2 i + 1), turned by position times frequency."""
    half = len(freq)
    ang = torch.arange(x.shape[0], dtype=torch.float64, device=DEV)[:, None, None] * freq
    c, s = ang.cos(), ang.sin()
    if interleaved:
        u, v = x[..., 0 : 2 * half : 2], x[..., 1 : 2 * half : 2]
        turned = torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)
    else:
        u, v = x[..., :half], x[..., half : 2 * half]
        turned = torch.cat([u * c - v * s, v * c + u * s], -1)
    return torch.cat([turned, x[..., 2 * half :]], -1)


def _attend(q, k, v, scale, seen, sink=None, softcap=None):
    """q [T, H, D], k and v [T, G, ..] -> [T, H, E]; ``sink`` [H]: the score of one more place that has no value."""
    T, H = q.shape[:2]
    out = []
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h] @ k[:, g].T) * scale
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        s = s.masked_fill(~seen, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink[h].expand(T, 1)], 1)
        out.append(torch.softmax(s, -1)[:, :T] @ v[:, g])
    return torch.stack(out, 1)


def _conv(x, taps, bias=None):
    """Causal sum over the last taps, the last one on the current token."""
    K = taps.shape[1]
    wide = torch.cat([x.new_zeros(K - 1, x.shape[1]), x])
    y = sum(wide[j : j + len(x)] * taps[:, j] for j in range(K))
    return _silu(y if bias is None else y + bias)


def _decayed(q, k, v, decay):
    """S <- decay S + k v^T, o = S^T q, a token at a time; decay [T, H, D], or [H, 1] the same at every token."""
    S = q.new_zeros(q.shape[1], q.shape[2], v.shape[2])
    out = []
    for t in range(len(q)):
        S = S * (decay[t] if decay.dim() == 3 else decay)[..., None] + k[t][:, :, None] * v[t][:, None, :]
        out.append((q[t][:, None, :] @ S)[:, 0])
    return torch.stack(out)


class _Plain:
    def __init__(self, case, seed):
        self.case, self.seed = case, seed
        self.raw = _llama_raw(case) if case["model"] == "llama" else _design_raw(case)
        self.eps = self.raw["rms_norm_eps"] if case["model"] == "llama" else self.raw["norm"]["eps"]
        self.kept = {}

    def w(self, name, *shape):
        """A weight in 64 bits; those of a depth's worth stay, a model's embedding or expert is made when it is wanted."""
        t = self.kept.get(name)
        if t is None:
            t = _tensor(self.case, self.seed, name, shape)
            if sum(x.numel() * x.element_size() for x in self.kept.values()) < 40e9:
                self.kept[name] = t
        return t.double()

    def row(self, name, shape, ids, cut=slice(None)):
        if name not in self.kept:
            self.kept[name] = _tensor(self.case, self.seed, name, shape)
        return self.kept[name][torch.as_tensor(ids, device=DEV)][:, cut].double()

    def lin(self, x, name, out, bias=False):
        y = x @ self.w(name, out, x.shape[-1]).T
        return y + self.w(name + ".b", out) if bias else y

    def normed(self, x, name):
        return _rms(x, self.eps) * self.w(name, x.shape[-1])

    def logits(self, ids):
        return (self.llama if self.case["model"] == "llama" else getattr(self, self.case["model"]))(ids)

    def causal(self, T, window=0, chunk=0):
        i, j = torch.arange(T, device=DEV)[:, None], torch.arange(T, device=DEV)[None, :]
        seen = j <= i
        if window:
            seen = seen & (i - j < window)
        return seen & (i // chunk == j // chunk) if chunk else seen

    # -------------------------------------------------------------- Llama

    def llama(self, ids):
        c, T = self.raw, len(ids)
        W, H, G, D, F = c["hidden_size"], c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], c["intermediate_size"]
        sc = c["rope_scaling"]
        freq = _frequencies(D, c["rope_theta"], (sc["factor"], sc["low_freq_factor"], sc["high_freq_factor"], sc["original_max_position_embeddings"]))
        x, seen = self.row("model.embed_tokens.weight", (VOCAB, W), ids), self.causal(T)
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = self.normed(x, p + "input_layernorm.weight")
            q, k, v = (self.lin(h, p + f"self_attn.{n}_proj.weight", m * D).view(T, m, D) for n, m in (("q", H), ("k", G), ("v", G)))
            a = _attend(_rotate(q, freq), _rotate(k, freq), v, D**-0.5, seen)
            x = x + self.lin(a.reshape(T, H * D), p + "self_attn.o_proj.weight", W)
            h = self.normed(x, p + "post_attention_layernorm.weight")
            a = _silu(self.lin(h, p + "mlp.gate_proj.weight", F)) * self.lin(h, p + "mlp.up_proj.weight", F)
            x = x + self.lin(a, p + "mlp.down_proj.weight", W)
        return self.lin(self.normed(x[-1:], "model.norm.weight"), "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight", VOCAB)

    # -------------------------------------------------------------- shared by the designs

    def experts(self, h, p, mlp, one, sel, wt, first=0):
        """Sum of the chosen experts' answers and the shared expert's."""
        n, out = mlp["router"]["experts"], torch.zeros_like(h)
        for e in range(n):
            at, place = (sel == e).nonzero(as_tuple=True)
            if len(at):
                out[at] += wt[at, place][:, None] * one(h[at], f"{p}e{e}.", mlp["expert"]["ff"])
        same = ((sel >= n) * wt).sum(-1, keepdim=True)  # experts that return their input
        return out + same * h

    def clipped(self, h, p, ff, limit=7.0):
        g, u = self.lin(h, p + "gate", ff).clamp(max=limit), self.lin(h, p + "up", ff).clamp(-limit, limit)
        return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1), p + "down", h.shape[1])

    def gated(self, h, p, ff):
        return self.lin(_silu(self.lin(h, p + "gate", ff)) * self.lin(h, p + "up", ff), p + "down", h.shape[1])

    def side(self, x, ids, layer, names):
        dim, n = self.raw["token_side"]["dim"], len(self.raw["layers"])
        e = self.row("side.embed", (VOCAB, n * dim), ids, slice(layer * dim, layer * dim + dim))
        return self.normed(self.lin(_gelu(self.lin(x, names + "gate", dim)) * e, names + "proj", x.shape[1]), names + "norm")

    def latent(self, h, p, m, interleaved, sinks):
        T, H, D, R, E, C = len(h), m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        q, dkv = self.lin(h, p + "q", H * (D + R)).view(T, H, D + R), self.lin(h, p + "dkv", C + R)
        c, freq = self.normed(dkv[:, :C], p + "dkv.norm"), _frequencies(R, m["rot"]["base"])
        k_rot = _rotate(dkv[:, C:].view(T, 1, R), freq, interleaved)
        k = torch.cat([self.lin(c, p + "uk", H * D).view(T, H, D), k_rot.expand(T, H, R)], -1)
        q = torch.cat([q[..., :D], _rotate(q[..., D:], freq, interleaved)], -1)
        seen = self.causal(T, (m.get("mask") or {}).get("size", 0))
        return _attend(q, k, self.lin(c, p + "uv", H * E).view(T, H, E), m["scale"], seen, self.w(p + "sink", H) if sinks else None).reshape(T, H * E)

    # -------------------------------------------------------------- Vuzelix

    def delta(self, h, p, m):
        T, H, D, E = len(h), m["heads"], m["dim"], m["vdim"]
        q, k, v = (_conv(self.lin(h, p + n, H * d), self.w(p + n + ".conv", H * d, m["conv"])).view(T, H, d) for n, d in (("q", D), ("k", D), ("v", E)))
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
        q, k, beta = unit(q) * D**-0.5, unit(k), torch.sigmoid(self.lin(h, p + "b", H))
        a = self.lin(self.lin(h, p + "a1", RANKS["vuzelix"]), p + "a2", H * D) + self.w(p + "dt_bias", H * D)
        g = torch.exp(-torch.exp(self.w(p + "A_log", H)).view(1, H, 1) * _softplus(a).view(T, H, D))
        S, o = h.new_zeros(H, D, E), []
        for t in range(T):
            S = S * g[t][..., None]
            u = beta[t][:, None] * (v[t] - (k[t][:, None, :] @ S)[:, 0])
            S = S + k[t][:, :, None] * u[:, None, :]
            o.append((q[t][:, None, :] @ S)[:, 0])
        gate = torch.sigmoid(self.lin(self.lin(h, p + "g1", RANKS["vuzelix"]), p + "g2", H * E)).view(T, H, E)
        return self.lin((self.normed(torch.stack(o), p + "norm") * gate).reshape(T, H * E), p + "o", h.shape[1])

    def vuzelix(self, ids):
        c, T, W = self.raw, len(ids), self.raw["width"]
        n, mult, keys = c["streams"], c["residual_mult"], {}
        xs = [self.row("embed", (VOCAB, W), ids)] * n

        def sublayer(xs, l, which, fn):
            name = f"l{l}.hc{which}."
            a, b, mix = self.w(name + "in", n), self.w(name + "out", n), self.w(name + "mix", n, n)
            y = fn(self.normed(sum(a[s] * xs[s] for s in range(n)), f"l{l}.norm{which}"))
            return [sum(mix[s, t] * xs[s] for s in range(n)) + mult * b[t] * y for t in range(n)]

        def attention(h, l, p, m):
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            own = m.get("kv_from") is None
            if own:
                keys[l] = _rms(self.lin(h, p + "k", G * D).view(T, G, D), self.eps), self.lin(h, p + "v", G * D).view(T, G, D)
            k, v = keys[l if own else m["kv_from"]]
            q = _rms(self.lin(h, p + "q", H * D).view(T, H, D), self.eps)
            o = _attend(q, k, v, m["scale"], self.causal(T, chunk=m["mask"]["size"]), h.new_zeros(H), m["softcap"])
            return self.lin(o.reshape(T, H * D), p + "o", W)

        for l, layer in enumerate(c["layers"]):
            m, p = layer["mixer"], f"l{l}.mix."
            xs = sublayer(xs, l, 1, lambda h: self.delta(h, p, m) if layer["type"] == "channel_delta" else attention(h, l, p, m))
            xs = sublayer(xs, l, 2, lambda h: self.lin(_gelu(self.lin(h, f"l{l}.mlp.up", layer["mlp"]["ff"])), f"l{l}.mlp.down", W))
        z = self.lin(self.normed(sum(xs)[-1:], "final.norm"), "head", VOCAB)
        return c["logit_softcap"] * torch.tanh(z / c["logit_softcap"])

    # -------------------------------------------------------------- Padetar

    def memory(self, h, p, m):
        T, H, D, E, cap = len(h), m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k, v = self.lin(h, p + "q", H * D).view(T, H, D) * D**-0.5, self.lin(h, p + "k", H * D).view(T, H, D), self.lin(h, p + "v", H * E).view(T, H, E)
        i = cap * torch.tanh(self.lin(h, p + "i", H, True) / cap)
        f = -_softplus(-cap * torch.tanh(self.lin(h, p + "f", H, True) / cap))
        S, n, top, out = h.new_zeros(H, D, E), h.new_zeros(H, D), h.new_zeros(H), []
        for t in range(T):
            new = torch.maximum(f[t] + top, i[t])
            a, b = torch.exp(f[t] + top - new), torch.exp(i[t] - new)
            bk = b[:, None] * k[t]
            S, n, top = a[:, None, None] * S + bk[:, :, None] * v[t][:, None, :], a[:, None] * n + bk, new
            den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
            out.append((q[t][:, None, :] @ S)[:, 0] / den[:, None])
        o = _rms(torch.stack(out), self.eps).reshape(T, H * E) * self.w(p + "norm", H * E)
        return self.lin(o * torch.sigmoid(self.lin(h, p + "g", H * E)), p + "o", h.shape[1])

    def padetar(self, ids):
        T, W = len(ids), self.raw["width"]
        x, seen = self.row("embed", (VOCAB, W), ids), self.causal(T)
        for l, layer in enumerate(self.raw["layers"]):
            p, m, mlp = f"l{l}.mix.left.", layer["mixer"]["left"], layer["mlp"]
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            sc = m["rot"]["scaling"]
            freq = _frequencies(D, m["rot"]["base"], (sc["factor"], sc["low"], sc["high"], sc["original"]))
            q, v = self.lin(x, p + "q", H * D, True).view(T, H, D), self.lin(x, p + "k", G * D, True).view(T, G, D)
            a = _attend(_rotate(self.normed(q, p + "q.norm"), freq), _rotate(self.normed(v, p + "k.norm"), freq), v, m["scale"], seen)
            y = self.lin(a.reshape(T, H * D), p + "o", W, True) + self.memory(x, f"l{l}.mix.right.", layer["mixer"]["right"])
            x = x + self.normed(y, f"l{l}.norm1")
            p = f"l{l}.mlp."
            val, sel = self.lin(x, p + "router", mlp["router"]["experts"], True).topk(mlp["router"]["top"], -1)
            y = self.experts(x, p, mlp, self.clipped, sel, torch.softmax(val, -1)) + self.clipped(x, p + "shared.", mlp["shared"]["ff"])
            x = x + self.normed(y, f"l{l}.norm2")
            x = x + self.side(x, ids, l, f"l{l}.side.")
        return self.lin(self.normed(x[-1:], "final.norm"), "head", VOCAB)

    # -------------------------------------------------------------- Fimilorn

    def fimilorn(self, ids):
        T, W = len(ids), self.raw["width"]
        first = x = self.row("embed", (VOCAB, W), ids)
        for l, enters in _order(self.raw):
            layer, p = self.raw["layers"][l], f"l{l}.mix."
            m, mlp = layer["mixer"], layer["mlp"]
            if enters is not None:
                x = x + (first if enters else 0.0) + self.w("loop.step", self.raw["loop"]["times"], W)[enters]
            h = self.normed(x, f"l{l}.norm1")
            if layer["type"] == "latent_attention":
                y = self.latent(h, p, m, False, True)
            else:
                H, G, D, E = m["heads"], m.get("kv_heads", m["heads"]), m["dim"], m["vdim"]
                q, k, v, g = self.lin(h, p + "q", H * D), self.lin(h, p + "k", G * D), self.lin(h, p + "v", G * E).view(T, G, E), self.lin(h, p + "g", H * E)
                freq = _frequencies(D, m["rot"]["base"])
                if layer["type"] == "attention":
                    q, k = self.normed(q, p + "q.norm"), self.normed(k, p + "k.norm")
                q, k = _rotate(q.view(T, H, D), freq), _rotate(k.view(T, G, D), freq)
                if layer["type"] == "attention":
                    y = _attend(q, k, v, m["scale"], self.causal(T), self.w(p + "sink", H)).reshape(T, H * E) * torch.sigmoid(g)
                else:
                    decay = torch.tensor(m["decay"], dtype=torch.float64, device=DEV)[:, None]
                    y = _rms(_decayed(q, k * D**-0.5, v, decay), self.eps).reshape(T, H * E) * _silu(g)
            x = x + self.normed(self.lin(y, p + "o", W), f"l{l}.norm1b")
            h, p = self.normed(x, f"l{l}.norm2"), f"l{l}.mlp."
            if mlp["kind"] == "dense":
                y = self.clipped(h, p, mlp["ff"], mlp["limit"])
            else:
                r = mlp["router"]
                s = torch.sigmoid(self.lin(h, p + "router", r["experts"]))
                by = (s + self.w(p + "correction", r["experts"])).view(T, r["groups"]["count"], -1)
                kept = by.topk(2, -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
                allow = torch.zeros(by.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, kept, True)
                sel = by.masked_fill(~allow[:, :, None], float("-inf")).reshape(T, -1).topk(r["top"], -1).indices
                y = self.experts(h, p, mlp, self.gated, sel, s.gather(1, sel)) + self.gated(h, p + "shared.", mlp["shared"]["ff"])
            x = x + self.normed(y, f"l{l}.norm2b")
        return self.lin(self.normed(x[-1:], "final.norm"), "embed", VOCAB)

    # -------------------------------------------------------------- Zipedra

    def zipedra(self, ids):
        T, W = len(ids), self.raw["width"]
        relu2 = lambda h, p, ff: self.lin(self.lin(h, p + "up", ff).clamp(min=0) ** 2, p + "down", W)
        first = x = self.row("embed", (VOCAB, W), ids)
        for l, enters in _order(self.raw):
            layer, p = self.raw["layers"][l], f"l{l}.mix."
            m, mlp = layer["mixer"], layer["mlp"]
            if enters is not None:
                x = self.lin(torch.cat([x, first], -1), "loop.in", W) + self.w("loop.step", self.raw["loop"]["times"], W)[enters]
            h = self.normed(x, f"l{l}.norm1")
            if layer["type"] == "latent_attention":
                y = self.latent(h, p, m, True, False)
            else:
                H, D, E = m["heads"], m["dim"], m["vdim"]
                q, k, v = (_silu(self.lin(h, p + n, H * d)).view(T, H, d) for n, d in (("q", D), ("k", D), ("v", E)))
                decay = torch.tensor(m["decay"], dtype=torch.float64, device=DEV)[:, None]
                y = self.normed(_decayed(q, k, v, decay).reshape(T, H * E), p + "norm")
            y = self.lin(y * torch.sigmoid(self.lin(h, p + "g", y.shape[1])), p + "o", W)
            p = f"l{l}.mlp."
            if mlp["kind"] == "dense":
                y = y + self.gated(h, p, mlp["ff"])
            else:
                s, sel = torch.softmax(self.lin(h, p + "router", mlp["router"]["experts"]), -1).topk(mlp["router"]["top"], -1)
                y = y + self.experts(h, p, mlp, relu2, sel, s / s.sum(-1, keepdim=True))
                y = y + torch.sigmoid(self.lin(h, p + "shared.sg", 1)) * relu2(h, p + "shared.", mlp["shared"]["ff"])
            x = x + y
            x = x + self.side(x, ids, l, f"l{l}.side.")
        return self.lin(self.normed(x[-1:], "final.norm"), "head", VOCAB) * self.raw["logit_scale"]

    # -------------------------------------------------------------- Meropel

    def selective(self, h, p, m):
        T, I, N, R = len(h), m["inner"], m["state"], m["dt_rank"]
        xz = self.lin(h, p + "in", 2 * I)
        x = _conv(xz[:, :I], self.w(p + "conv", I, m["conv"]), self.w(p + "conv.b", I))
        dbc = self.lin(x, p + "x", R + 2 * N)
        dt = _softplus(self.lin(dbc[:, :R], p + "dt", I, True))
        A, S, y = -torch.exp(self.w(p + "A_log", I, N)), h.new_zeros(I, N), []
        for t in range(T):
            S = S * torch.exp(dt[t][:, None] * A) + (dt[t] * x[t])[:, None] * dbc[t, R : R + N]
            y.append(S @ dbc[t, R + N :])
        return self.lin((torch.stack(y) + self.w(p + "D", I) * x) * _silu(xz[:, I:]), p + "o", h.shape[1])

    def mamba2(self, h, p, m):
        T, H, E, N = len(h), m["heads"], m["vdim"], m["state"]
        I = H * E
        zxd = self.lin(h, p + "in", 2 * I + 2 * N + H)
        xbc = _conv(zxd[:, I : 2 * I + 2 * N], self.w(p + "conv", I + 2 * N, m["conv"]), self.w(p + "conv.b", I + 2 * N))
        dt = _softplus(zxd[:, 2 * I + 2 * N :] + self.w(p + "dt_bias", H))
        x, B, C = xbc[:, :I].view(T, H, E), xbc[:, None, I : I + N].expand(T, H, N), xbc[:, None, I + N :].expand(T, H, N)
        decay = torch.exp(-torch.exp(self.w(p + "A_log", H)) * dt)[..., None]
        y = _decayed(C, dt[..., None] * B, x, decay) + self.w(p + "D", H)[:, None] * x
        return self.lin(self.normed(y.reshape(T, I) * _silu(zxd[:, :I]), p + "norm"), p + "o", h.shape[1])

    def meropel(self, ids):
        T, W = len(ids), self.raw["width"]
        b = self.raw["embedding"]["bigram"]
        pairs = [b["buckets"]] + [(u * b["mul_prev"] + v * b["mul_cur"]) % b["buckets"] for u, v in zip(ids, ids[1:])]
        x = self.row("embed", (VOCAB, W), ids) + self.row("bigram", (b["buckets"] + 1, W), pairs)
        seen = self.causal(T)
        for l, layer in enumerate(self.raw["layers"]):
            p, m, mlp = f"l{l}.mix.", layer["mixer"], layer["mlp"]
            h = self.normed(x, f"l{l}.norm1")
            if layer["type"] == "gla":
                H, D, E = m["heads"], m["dim"], m["vdim"]
                q, k, v = (self.lin(h, p + n, H * d).view(T, H, d) for n, d in (("q", D), ("k", D), ("v", E)))
                z = self.lin(self.lin(h, p + "a1", RANKS["meropel"]), p + "a2", H * D, True)
                o = self.normed(_decayed(q * D**-0.5, k, v, torch.exp(-_softplus(-z) / m["tau"]).view(T, H, D)), p + "norm")
                y = self.lin(o.reshape(T, H * E) * _silu(self.lin(h, p + "g", H * E)), p + "o", W)
            else:
                a, two = m["left"], layer["type"] == "parallel_2"
                H, G, D, E = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
                q, k, v = (self.lin(h, p + "left." + n, d, two) for n, d in (("q", H * D), ("k", G * D), ("v", G * E)))
                if two:
                    q, k = self.normed(q, p + "left.q.norm"), self.normed(k, p + "left.k.norm")
                freq = _frequencies(a["rot"]["dims"], a["rot"]["base"])
                o = _attend(_rotate(q.view(T, H, D), freq, two), _rotate(k.view(T, G, D), freq, two), v.view(T, G, E), a["scale"], seen)
                if two:
                    left, right = self.lin(o.reshape(T, H * E), p + "left.o", W), self.mamba2(h, p + "right.", m["right"])
                    y = 0.5 * (self.normed(left, p + "left.out") + self.normed(right, p + "right.out"))
                else:
                    o = o * torch.sigmoid(self.lin(h, p + "left.g", H))[:, :, None]
                    y = self.lin(o.reshape(T, H * E), p + "left.o", W) + self.selective(h, p + "right.", m["right"])
            x = x + self.normed(y, f"l{l}.norm1b")
            h, p = self.normed(x, f"l{l}.norm2"), f"l{l}.mlp."
            if mlp["kind"] == "dense":
                y = self.gated(h, p, mlp["ff"])
            else:
                r = mlp["router"]
                n = r["experts"] + r["identity"]
                s = torch.softmax(self.lin(h, p + "router", n), -1)
                by = (s + self.w(p + "correction", n)).view(T, r["groups"]["count"], -1)
                kept = by.amax(-1).topk(r["groups"]["keep"], -1).indices
                allow = torch.zeros(by.shape[:2], dtype=torch.bool, device=DEV).scatter_(1, kept, True)
                sel = by.masked_fill(~allow[:, :, None], float("-inf")).reshape(T, -1).topk(r["top"], -1).indices
                wt = s.gather(1, sel)
                y = self.experts(h, p, mlp, self.gated, sel, wt / wt.sum(-1, keepdim=True) * r["scale"]) + self.gated(h, p + "shared.", mlp["shared"]["ff"])
            x = x + self.normed(y, f"l{l}.norm2b")
        return self.lin(self.normed(x[-1:], "final.norm"), "head", VOCAB) * self.raw["logit_scale"]
