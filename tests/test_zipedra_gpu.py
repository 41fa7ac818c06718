"""The Zipedra design in the framework against the plain implementation of ``plain_zipedra``: every mechanism alone at
sizes of its own, then whole models through the step function, the cache and state manager, the scheduler and the
engine, for the same requests cut into steps in different ways.  Configurations and weights are made here."""

from __future__ import annotations

import json
import random

import pytest
import torch

import plain_zipedra as pz
import traces
from harness import batch, close, counted, in_long_portions, paged, replay, step_context
from tiny import random_tokens

pytestmark = pytest.mark.gpu
DEV = "cuda"
BOTH = pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])


def latent(H, D, R, E, C, scale, base=50000.0):
    return "latent_attention", dict(heads=H, dim=D, rot_dim=R, vdim=E, kv_rank=C, scale=scale, rot={"base": base, "dims": R})


def lightning(H, D, E, decay):
    return "lightning", dict(heads=H, dim=D, vdim=E, decay=list(decay))


def dense(ff):
    return {"kind": "dense", "ff": ff}


def moe(n, top, ff, shared=0):
    out = {"kind": "moe", "expert": {"ff": ff}, "router": {"experts": n, "top": top}}
    if shared:
        out["shared"] = {"ff": shared}
    return out


def layer(mixer, mlp):
    return {"type": mixer[0], "mixer": mixer[1], "mlp": mlp}


# A: sizes that are no multiples of 8 or 16 (a width that is no multiple of four), a layer without feed-forward, experts with
#    and without a shared one, the middle layers run three times with a layer in front of them and one behind.
# B: one head everywhere, one expert of one, no loop and no token input (both sublayers' outputs wait for the next layer's
#    read), no logit scale, one rotated pair, a head that never forgets.
# C: sizes the matrix-core kernels take in bfloat16, all layers run twice, all experts chosen in one of them.
# D: latent layers whose long prompt portions have keys and values of their own made (both sets of sizes).
CONFIGS = {
    "A": dict(cfg={"architecture": "Zipedra", "vocab": 300, "width": 90, "norm": {"eps": 1e-5}, "logit_scale": 0.5, "token_side": {"dim": 7},
                   "loop": {"start": 1, "stop": 3, "times": 3},
                   "layers": [layer(latent(3, 12, 6, 10, 24, 0.3, base=5000.0), dense(50)),
                              layer(lightning(3, 10, 22, (0.9, 0.97, 0.995)), moe(6, 3, 20, shared=28)),
                              layer(latent(2, 20, 4, 6, 18, 0.35), None),
                              layer(lightning(1, 24, 6, (0.99,)), moe(5, 2, 24))]},
              seed=3, page=8, lengths=(1, 2, 23, 77, 150, 203)),
    "B": dict(cfg={"architecture": "Zipedra", "vocab": 128, "width": 64, "norm": {"eps": 1e-6},
                   "layers": [layer(latent(1, 16, 2, 24, 16, 0.4, base=100.0), moe(1, 1, 48)),
                              layer(lightning(1, 64, 8, (1.0,)), dense(40)),
                              layer(lightning(2, 8, 16, (0.5, 0.999)), None)]},
              seed=4, page=16, lengths=(3, 8, 9, 40, 129)),
    "C": dict(cfg={"architecture": "Zipedra", "vocab": 200, "width": 128, "norm": {"eps": 1e-5}, "logit_scale": 2.0, "token_side": {"dim": 16},
                   "loop": {"start": 0, "stop": 3, "times": 2},
                   "layers": [layer(latent(4, 32, 32, 64, 96, 0.15, base=1e6), moe(4, 4, 64, shared=96)),
                              layer(lightning(4, 32, 48, (0.9, 0.95, 0.99, 0.999)), dense(256)),
                              layer(lightning(2, 64, 32, (0.8, 0.97)), moe(16, 3, 32, shared=64))]},
              seed=5, page=16, lengths=(5, 31, 64, 100, 260)),
    "D": dict(cfg={"architecture": "Zipedra", "vocab": 200, "width": 128, "norm": {"eps": 1e-5}, "logit_scale": 2.0,
                   "layers": [layer(latent(4, 64, 32, 64, 128, 0.15, base=1e6), moe(8, 2, 64, shared=96)),
                              layer(latent(2, 128, 64, 128, 128, 0.1), dense(256))]},
              seed=6, page=16, lengths=(3, 27, 130, 260, 400)),
}
# what random weights of the usual law leave so small that soft-maxes are flat, gates constant and SiLUs linear (the first
# tail of a name that fits)
SHARPEN = {"side.embed": 25.0, "embed": 25.0, "side.gate": 6.0, "side.proj": 6.0, "mix.q": 6.0, "mix.k": 6.0, "mix.v": 6.0, "mix.g": 8.0, "mix.uk": 6.0,
           "mix.uv": 4.0, "mix.o": 3.0, "router": 10.0, ".sg": 8.0, ".gate": 6.0, ".up": 6.0, ".down": 3.0, "loop.in": 4.0, "loop.step": 10.0}


def write_folder(folder, cfg: dict, seed: int, change=None):
    """config.json and model.safetensors with random 32-bit weights for the tensors the framework says the model reads."""
    from safetensors.torch import save_file

    from nanospec_amd.config import ZipedraConfig
    from nanospec_amd.parts.model import wanted_tensors
    from nanospec_amd.weights import random_tensors

    folder.mkdir(parents=True, exist_ok=True)
    tensors = random_tensors(wanted_tensors(ZipedraConfig.from_hf(cfg).model_spec()), seed, torch.float32)
    for name, t in tensors.items():
        t *= next((by for tail, by in SHARPEN.items() if name.endswith(tail)), 1.0)
    if change is not None:
        change(tensors)
    (folder / "config.json").write_text(json.dumps(cfg))
    save_file({k: v.contiguous() for k, v in tensors.items()}, str(folder / "model.safetensors"))
    return folder


@pytest.fixture(scope="module")
def folders(tmp_path_factory):
    base = tmp_path_factory.mktemp("zipedra")
    return {name: write_folder(base / name, c["cfg"], c["seed"]) for name, c in CONFIGS.items()}


def read_folder(folder, dtype):
    from safetensors.torch import load_file

    cfg = json.loads((folder / "config.json").read_text())
    w = {k: v.to(dtype).double() for k, v in load_file(str(folder / "model.safetensors")).items()}  # as the engine rounds them
    return cfg, w


def sequences(name):
    c = CONFIGS[name]
    return {f"r{i}": random_tokens(n, c["cfg"]["vocab"], 31 * i + n) for i, n in enumerate(c["lengths"])}


_REF, _MODELS = {}, {}


def plain_logits(folder, name, dtype):
    if (name, dtype) not in _REF:
        cfg, w = read_folder(folder, dtype)
        _REF[name, dtype] = {rid: pz.forward(cfg, w, toks).float() for rid, toks in sequences(name).items()}
    return _REF[name, dtype]


def engine_model(folder, name, dtype):
    from nanospec_amd.loader import load_model

    if (name, dtype) not in _MODELS:
        _MODELS[name, dtype] = load_model(folder, dtype=dtype)
    return _MODELS[name, dtype]


class Ctx:
    """The little that a part without a cache asks of a step's context."""

    captured = False

    def __init__(self):
        from nanospec_amd.engine.arena import Arena

        self.arena, self.plans = Arena(torch.device(DEV)), {}

    def requests(self, lens, slots, positions, plan=None, spare=0):
        """A batch of hand-made requests; ``plan``: a batch plan that describes it, in a region of ``spare`` more entries than it needs."""
        import types

        import numpy as np

        self.token_req, self.qo_indptr, self.state_slots = batch(lens, slots)
        self.positions = torch.tensor(positions, dtype=torch.int32, device=DEV)
        self.max_position = max(positions)
        if plan is not None:
            shape = plan.shape(lens)
            shape = (shape[0] + spare, *shape[1:])
            out = np.full(max(1, plan.ints(shape)), -1, dtype=np.int32)
            plan.fill(out, shape, types.SimpleNamespace(covered=len(lens), lens=np.array(lens), indptr=np.concatenate([[0], np.cumsum(lens)])))
            self.plans = {plan.key: (torch.from_numpy(out).to(DEV), shape)}


def off(got, want):
    """The largest difference over the largest value, and the root mean square of the difference over that of the values."""
    d = got.cpu().double() - want
    return float(d.abs().max() / want.abs().max()), float(d.pow(2).mean().sqrt() / want.pow(2).mean().sqrt())


# ------------------------------------------------------------------------------------------------ whole models


@BOTH
@pytest.mark.parametrize("name", list(CONFIGS))
@pytest.mark.parametrize("schedule", ["whole", "tail", "portions", "mixed", "mixed7"])
def test_schedules_match_plain(folders, name, dtype, schedule):
    """Whole prompts; prefill then token-by-token decoding (120 tokens, through captured steps); portions down to two
    tokens; mixed batches of unequal requests in a pool so small that pages and state slots are used again."""
    page = CONFIGS[name]["page"]
    seqs, ref, model = sequences(name), plain_logits(folders[name], name, dtype), engine_model(folders[name], name, dtype)
    longest = max(len(t) for t in seqs.values())
    if schedule == "whole":
        steps, where = traces.whole(seqs)
    elif schedule == "tail":
        steps, where = traces.tail_decoded(seqs, tail=120)
    elif schedule == "portions":
        steps, where = traces.portions(seqs, seed=1)
    else:
        steps, where, peak = traces.mixed(seqs, seed=7 if schedule == "mixed7" else 0, max_live=2 if schedule == "mixed7" else 3)
    max_tokens = peak if schedule.startswith("mixed") else -(-longest // 64) * 64
    rep = replay(model, steps, where, ref, dtype, max_tokens, page)
    if schedule.startswith("mixed"):
        assert rep.pages_again > 0 and rep.slots_again > 0, "the pool was meant to hand pages and slots out again"
    if schedule == "tail":
        assert rep.graph_steps > 0, "single decoded tokens were meant to replay captured steps"


@BOTH
@pytest.mark.parametrize("name", list(CONFIGS))
def test_the_stream_after_every_layer(folders, name, dtype):
    """The residual stream after each layer that runs (a layer of the range that runs several times counts each time), not
    only the logits: a fault shows in the layer that has it."""
    from nanospec_amd.engine.replay import Replayer

    model = engine_model(folders[name], name, dtype)
    cfg, w = read_folder(folders[name], dtype)
    toks = sequences(name)["r3"]
    ref, got = [], []
    pz.forward(cfg, w, toks, probe=lambda run, x: ref.append(x.clone()))
    model.layer_probe = lambda i, total: got.append(total.clone())
    try:
        Replayer(model, 256, page_size=CONFIGS[name]["page"], use_graphs=False).step([{"id": "a", "tokens": toks, "want": [0]}], ["a"])
    finally:
        model.layer_probe = None
    assert len(got) == len(pz.run_order(cfg)) == len(ref)
    for i, g in enumerate(got):
        err = (g.cpu() - ref[i].float()).abs().amax(-1) / ref[i].abs().max()
        if dtype == torch.float32:
            assert err.max() <= 2e-5, f"after layer run {i}: {err.max():.2e}"
        else:  # (a token may take another expert where two router scores lie within rounding of each other)
            assert (err > 0.1).sum() <= max(2, len(toks) // 10) and err.median() <= 0.03, f"after layer run {i}: {err}"


@BOTH
@pytest.mark.parametrize("name", list(CONFIGS))
def test_one_position_however_it_is_reached(folders, name, dtype):
    """The logits at one position are the same (beyond rounding) whole, decoded, in portions cut at and around the pages'
    edges and the recurrence's blocks of tokens, and beside other requests."""
    from nanospec_amd.engine.replay import Replayer

    model, seqs = engine_model(folders[name], name, dtype), sequences(name)
    toks = seqs["r4"]
    last = len(toks) - 1
    rep = Replayer(model, 1024, page_size=CONFIGS[name]["page"])
    got = [rep.step([{"id": "w", "tokens": toks, "want": [last]}], ["w"])[0]]
    rep.step([{"id": "d", "tokens": toks[:-1], "want": []}], [])
    got.append(rep.step([{"id": "d", "tokens": toks[-1:], "want": [0]}], ["d"])[0])
    cuts = [0, 2, 4, 5, 7, 8, 9, 10, 15, 16, 17, 23, 24, 26, 63, 64, 65, 113, last - 9, last - 8, last - 5, last - 4, last - 1, len(toks)]
    cuts = sorted({c for c in cuts if 0 <= c <= len(toks)})
    other = seqs["r3"]
    for a, b in zip(cuts, cuts[1:]):
        entries = [{"id": "p", "tokens": toks[a:b], "want": [b - a - 1]}]
        if a < len(other):
            entries.insert(0, {"id": "o", "tokens": other[a : min(b, len(other))], "want": []})
        out = rep.step(entries, ["p"] if b == len(toks) else [])
    got.append(out[-1])
    tol = 2e-5 if dtype == torch.float32 else 0.08
    for g in got[1:]:
        assert (g - got[0]).abs().max() <= tol * got[0].abs().max()


@BOTH
def test_long_portions_beside_decoded_tokens_through_captured_steps(folders, dtype):
    """A portion long enough for the recurrence's chunks beside single tokens of another request, in one captured shape that is
    replayed with other requests and other lengths (long portions, a short one that the scan takes, none)."""
    from nanospec_amd.engine.replay import Replayer

    model, seqs, ref = engine_model(folders["C"], "C", dtype), sequences("C"), plain_logits(folders["C"], "C", dtype)
    long, short = seqs["r4"], seqs["r3"]
    rep = Replayer(model, 512, page_size=CONFIGS["C"]["page"])
    rep.step([{"id": "d", "tokens": short[:40], "want": []}], [])
    at, loose, rows = 40, [], 0
    for trial, cuts in enumerate(([0, 200, 205, 260], [0, 250, 258], [0, 60, 259], [0, 195, 198])):
        for a, b in zip(cuts, cuts[1:]):
            end = b == cuts[-1]
            out = rep.step([{"id": "d", "tokens": [short[at]], "want": [0]}, {"id": f"p{trial}", "tokens": long[a:b], "want": [0, b - a - 1]}],
                           [f"p{trial}"] if end else [])
            assert rep.runner.last_used_graph, "the step was meant to replay a captured graph"
            close(out, torch.stack([ref["r3"][at], ref["r4"][a], ref["r4"][b - 1]]), dtype, (trial, a, b), loose)
            at, rows = at + 1, rows + 3
    assert len(loose) <= max(2, rows // 10), loose


@pytest.mark.parametrize("graphs", [False, True], ids=["eager", "captured"])
def test_long_portions_of_latent_layers(folders, monkeypatch, graphs):
    """Portions over keys and values made from the latents, beside single tokens over the latents themselves, and one after the other for
    the same request."""
    from nanospec_amd.kernels import ops

    dtype, loose = torch.bfloat16, []
    model, have, ref = engine_model(folders["D"], "D", dtype), sequences("D"), plain_logits(folders["D"], "D", dtype)
    names = {"s": "r1", "m": "r3", "l": "r4"}
    in_long_portions(model, {k: have[r] for k, r in names.items()}, {k: ref[r] for k, r in names.items()},
                     lambda got, want, what: close(got, want, dtype, what, loose), CONFIGS["D"]["page"], graphs, counted(monkeypatch, ops, "latent_prompt"))
    assert len(loose) <= 8, loose  # (of 82 rows, each counted twice: a token may take another expert)


def test_long_decoding_keeps_the_state(folders):
    """400 tokens one by one after a short prompt, in 32-bit: the lightning layers' state (one head never forgets) and the
    latent layers' pages carry every token; the last logits are those of the whole sequence at once."""
    cfg, w = read_folder(folders["B"], torch.float32)
    toks = random_tokens(420, cfg["vocab"], 99)
    ref = {"a": pz.forward(cfg, w, toks).float()}
    steps, where = traces.tail_decoded({"a": toks}, tail=400)
    replay(engine_model(folders["B"], "B", torch.float32), steps, where, ref, torch.float32, 448, CONFIGS["B"]["page"])


@BOTH
@pytest.mark.parametrize("name", ["A", "B"])
def test_greedy_generation_through_the_engine(folders, name, dtype):
    """``Engine.generate`` with a token budget and a longest portion, so that the scheduler cuts prompts and batches portions
    beside decoding requests; against the plain implementation's greedy continuation (in bfloat16 a sequence may leave it
    only where the plain logits of the two tokens are within rounding of each other)."""
    from nanospec_amd import Engine, EngineConfig, SamplingParams

    page = CONFIGS[name]["page"]
    model = engine_model(folders[name], name, dtype)
    cfg, w = read_folder(folders[name], dtype)
    prompts = [t for t in sequences(name).values() if len(t) < 100][:4]
    new = 12
    eng = Engine(model, EngineConfig(num_blocks=sum(-(-(len(p) + new) // page) for p in prompts) + 2, block_size=page, max_step_tokens=48,
                                     prefill_chunk=20, max_running=4))
    got = eng.generate(prompts, SamplingParams(max_tokens=new))
    eng.cache.check()
    for prompt, ours in zip(prompts, got):
        seq = list(prompt)
        for k, tok in enumerate(ours):
            row = pz.forward(cfg, w, seq)[-1]
            best = int(row.argmax())
            if tok != best:
                gap = float(row[best] - row[tok]) / float((row - row.mean()).pow(2).mean().sqrt())
                assert dtype == torch.bfloat16 and gap < 0.25, f"{name} {dtype}: token {k} is {tok}, plain {best} (gap {gap:.3f})"
                break
            seq.append(tok)
        assert len(ours) == new


def test_preempted_requests_start_their_state_again(folders):
    """A pool too small for all requests with the policy that releases the newest one and recomputes it later: its state
    starts from zero at its second admission, and the tokens are those of a pool that is large enough."""
    from nanospec_amd import Engine, EngineConfig, SamplingParams

    page = CONFIGS["A"]["page"]
    model = engine_model(folders["A"], "A", torch.float32)
    prompts = [t[:20] for t in sequences("A").values() if len(t) >= 20] * 2
    new = 30
    calm = Engine(model, EngineConfig(num_blocks=128, block_size=page)).generate(prompts, SamplingParams(max_tokens=new))
    eng = Engine(model, EngineConfig(num_blocks=23, block_size=page, on_exhaustion="preempt", prefill_chunk=16))
    rough = eng.generate(prompts, SamplingParams(max_tokens=new))
    assert eng.sched.preempted_total > 0, "the pool was meant to run out"
    assert rough == calm
    eng.cache.check()


def test_the_command_lines_generate_and_replay(folders, tmp_path):
    """``python -m nanospec_amd`` continues a prompt greedily; ``bin/trace_run`` replays two steps of the same model."""
    import subprocess
    import sys
    from pathlib import Path

    import numpy as np

    root = Path(__file__).resolve().parent.parent
    out = subprocess.run([sys.executable, "-m", "nanospec_amd", "--model", str(folders["B"]), "--prompt-ids", "1,2,3,4,5", "--max-tokens", "4",
                          "--dtype", "float32", "--block-size", "16"], cwd=root, capture_output=True, text=True, timeout=300)
    assert out.returncode == 0, out.stderr[-2000:]
    row = json.loads(out.stdout.strip().splitlines()[-1])
    cfg, w = read_folder(folders["B"], torch.float32)
    seq = [1, 2, 3, 4, 5]
    for tok in row["output_ids"]:
        assert tok == int(pz.forward(cfg, w, seq)[-1].argmax())
        seq.append(tok)
    assert len(row["output_ids"]) == 4
    steps = [{"step": 0, "entries": [{"id": "a", "tokens": [1, 2, 3], "want": [1]}], "end": []},
             {"step": 1, "entries": [{"id": "a", "tokens": [4, 5], "want": [0, 1]}], "end": ["a"]}]
    out = subprocess.run([str(root / "bin" / "trace_run"), "--model", str(folders["B"]), "--dtype", "float32", "--out", str(tmp_path), "--max-tokens", "64"],
                         input="\n".join(json.dumps(s) for s in steps) + "\n", capture_output=True, text=True, timeout=300)
    assert out.returncode == 0 and "done 1" in out.stdout.splitlines(), out.stderr[-2000:]
    ref = pz.forward(cfg, w, [1, 2, 3, 4, 5]).float()
    for step, rows in ((0, [1]), (1, [3, 4])):
        got = torch.from_numpy(np.fromfile(tmp_path / f"{step}.f32", dtype="<f4")).view(len(rows), -1)
        close(got, ref[rows], torch.float32, f"step {step}")


def drawn_config(seed: int) -> dict:
    """A configuration drawn from everything the design lets a model choose."""
    rng = random.Random(1000 + seed)
    layers = []
    for _ in range(rng.randint(1, 5)):
        D = rng.choice([8, 12, 24, 32, 40])
        if rng.random() < 0.5:
            H = rng.choice([1, 2, 5])
            mixer = lightning(H, D, rng.choice([5, 16, 40]), [rng.choice([0.5, 0.9, 0.99, 0.999, 1.0]) for _ in range(H)])
        else:
            mixer = latent(rng.choice([1, 2, 5]), D, rng.choice([2, 8, 16]), rng.choice([8, 20, 48]), rng.choice([8, 24, 32]), rng.uniform(0.1, 0.5),
                           base=rng.choice([100.0, 1e4]))
        r = rng.random()
        n = rng.choice([2, 4, 7])
        mlp = None if r < 0.2 else (dense(rng.choice([8, 20, 48])) if r < 0.45 else moe(n, rng.randint(1, n), rng.choice([8, 20, 48]), rng.choice([0, 8, 40])))
        layers.append(layer(mixer, mlp))
    cfg = {"architecture": "Zipedra", "vocab": rng.choice([50, 128, 333]), "width": rng.choice([32, 50, 64, 100, 136]),
           "norm": {"eps": rng.choice([1e-6, 1e-5, 1e-3])}, "logit_scale": rng.choice([0.3, 1.0]), "layers": layers}
    if rng.random() < 0.7:
        cfg["token_side"] = {"dim": rng.choice([1, 5, 16])}
    if rng.random() < 0.7:
        start = rng.randrange(len(layers))
        cfg["loop"] = {"start": start, "stop": rng.randint(start + 1, len(layers)), "times": rng.choice([1, 2, 3])}
    return cfg


@BOTH
@pytest.mark.parametrize("seed", range(8))
def test_drawn_configurations_match_plain(tmp_path, seed, dtype):
    """Eight configurations drawn at random: in portions, then in a mixed batch, in a small pool.  (Some of them choose one
    expert of two: there a close call that bfloat16 rounding moves changes a row altogether, so more rows may differ by more
    than rounding.)"""
    from nanospec_amd.loader import load_model

    folder = write_folder(tmp_path / "m", drawn_config(seed), seed)
    model = load_model(folder, dtype=dtype)
    cfg, w = read_folder(folder, dtype)
    seqs = {f"r{i}": random_tokens(n, cfg["vocab"], 7 * i + seed) for i, n in enumerate((1, 2, 19, 70, 131))}
    ref = {rid: pz.forward(cfg, w, toks).float() for rid, toks in seqs.items()}
    page = [4, 8, 16][seed % 3]
    steps, where = traces.portions(seqs, seed=seed)
    replay(model, steps, where, ref, dtype, 192, page, loose_share=5, caps=(0.2, 0.12))
    steps, where, peak = traces.mixed(seqs, seed=seed, max_live=3)
    replay(model, steps, where, ref, dtype, peak, page, loose_share=5, caps=(0.2, 0.12))


@BOTH
@pytest.mark.parametrize("mark", [0, 15, 16, 17, 131])
def test_a_far_key_decides_the_answer(folders, tmp_path, dtype, mark):
    """The first layer of model B is latent attention with one head.  Its query matrix is made minus its key path's (up to the
    latent's norm), its rotated query part zero, and two tokens get large embeddings of opposite sign: the query of the one at
    the end then meets the key of the other (and not its own), ``mark`` tokens into the sequence, with the largest score there
    can be, among hundreds of others.  The plain logits at the end change when that one token is taken away; the framework's
    follow them, in a prompt and decoded."""
    from nanospec_amd.loader import load_model

    m = CONFIGS["B"]["cfg"]["layers"][0]["mixer"]

    def change(w):
        q = torch.zeros_like(w["l0.mix.q"])
        q[: m["dim"]] = -60.0 * w["l0.mix.uk"] @ w["l0.mix.dkv"][: m["kv_rank"]]
        w["l0.mix.q"] = q
        w["l0.mix.o"] *= 8.0
        w["embed"][4] = torch.randn(w["embed"].shape[1], generator=torch.Generator().manual_seed(1))
        w["embed"][3] = -w["embed"][4]

    X, Y, Z = 3, 4, 5
    folder = write_folder(tmp_path / "far", CONFIGS["B"]["cfg"], CONFIGS["B"]["seed"], change)
    cfg, wd = read_folder(folder, dtype)
    toks = [t if t not in (X, Y) else Z for t in random_tokens(300, cfg["vocab"], 5)]
    toks[mark], toks[-1] = X, Y
    ref = pz.forward(cfg, wd, toks).float()
    without = pz.forward(cfg, wd, toks[:mark] + [Z] + toks[mark + 1 :]).float()[-1]
    spread = (ref[-1] - ref[-1].mean()).pow(2).mean().sqrt()
    assert (ref[-1] - without).pow(2).mean().sqrt() > 0.1 * spread, "the test's far key was meant to matter"
    model = load_model(folder, dtype=dtype)
    for tail in (1, 40):
        steps, where = traces.tail_decoded({"a": toks}, tail=tail)
        replay(model, steps, where, {"a": ref}, dtype, 320, CONFIGS["B"]["page"])


# ------------------------------------------------------------------------------------------------ mechanisms alone


def lightning_part(dtype, H, D, E, decay, W=48, eps=1e-5):
    """The mixer as the framework builds it from the design's configuration, with random weights -> (part, plain weights)."""
    from nanospec_amd.config import ZipedraConfig
    from nanospec_amd.config.zipedra import ZipedraLayer
    from nanospec_amd.parts import registry
    from nanospec_amd.weights import random_tensors

    spec = ZipedraConfig(vocab=8, width=W, layers=(), norm_eps=eps)._mixer(ZipedraLayer(type="lightning", heads=H, dim=D, vdim=E, decay=tuple(decay)))
    part = registry.build("mixer", spec, "")
    tensors = random_tensors(part.wanted(), H * D + E, torch.float32)
    assert set(tensors) == {"q", "k", "v", "g", "o", "norm"}
    for name in ("q", "k", "v", "g"):
        tensors[name] *= 15.0
    tensors = {k: v.to(dtype) for k, v in tensors.items()}
    part.load(lambda name: tensors[name], dtype, DEV)
    return part, {k: v.double() for k, v in tensors.items()}


@BOTH
@pytest.mark.parametrize("chunked", [False, True], ids=["scan", "chunks"])
@pytest.mark.parametrize("H,D,E", [(3, 20, 36), (1, 64, 8), (5, 9, 7), (4, 128, 256), (2, 16, 300), (1, 200, 40)])
def test_lightning_through_the_part(monkeypatch, dtype, H, D, E, chunked):
    """The mixer (stacked product, SiLUs, recurrence, the norm over all heads with the gate, output product) against the plain
    recurrence: three requests in state slots that are not in order, cut into unequal portions (one of them a token at a
    time, one with a portion of more than two chunks), each step finding the state that the step before left; a freed slot
    serves another request from zero.  Token by token, and with the long portions in chunks (where the key size allows it)."""
    from nanospec_amd.parts import retention
    from nanospec_amd.parts.retention import CHUNKS

    monkeypatch.setattr(retention, "CHUNKED_FROM", 64)
    W, eps = 48, 1e-5
    decay = [(0.5, 0.97, 1.0, 0.999, 0.9)[h % 5] for h in range(H)]
    part, w = lightning_part(dtype, H, D, E, decay)
    m = dict(heads=H, dim=D, vdim=E, decay=decay)
    g = torch.Generator().manual_seed(7)
    seqs = [torch.randn(n, W, generator=g).to(dtype) for n in (9, 5, 214, 70)]
    ref = [pz.lightning(s.double(), w, "", m, eps, torch.arange(len(s))) for s in seqs]
    slots = [4, 0, 2, 0]  # the last request takes the slot of the second after it has ended
    cuts = [[0, 4, 5, 9], [0, 1, 2, 3, 4, 5], [0, 2, 19, 150, 214]]
    state = torch.randn(6, H * D * E, device=DEV)  # what earlier requests left
    ctx = Ctx()
    plan = CHUNKS if chunked else None
    assert bool(part.batch_plans()) == (D % 4 == 0)

    def run(live, parts):
        x = torch.cat([seqs[b][a:e] for b, (a, e) in zip(live, parts)]).to(DEV)
        ctx.requests([e - a for a, e in parts], [slots[b] for b in live], [p for a, e in parts for p in range(a, e)], plan, spare=2)
        mark = ctx.arena.mark()
        y = part.forward(ctx, x, type("V", (), {"state": state})()).cpu()
        ctx.arena.release(mark)
        want = torch.cat([ref[b][a:e] for b, (a, e) in zip(live, parts)])
        worst, rms = off(y, want)
        assert worst <= 1e-4 if dtype == torch.float32 else rms <= 3e-2, (live, parts, worst, rms)

    for s in set(slots):
        state[s] = 0  # as at admission
    for step in range(5):
        live = [b for b in range(3) if step + 1 < len(cuts[b])]
        if live:
            run(live, [(cuts[b][step], cuts[b][step + 1]) for b in live])
    state[0] = 0
    run([3], [(0, 70)])


@pytest.mark.parametrize("H,D,E", [(2, 16, 24), (1, 128, 144), (4, 36, 65)])
@pytest.mark.parametrize("gap", [63, 64, 65, 127, 128, 200])
def test_chunks_read_back_what_the_first_token_wrote(monkeypatch, gap, H, D, E):
    """One key channel is written by the first token alone and read by the last one alone, ``gap`` tokens later: in the same
    portion, inside the chunk and across chunks, and in the portion behind it.  The read-out is the first token's value times
    decay^gap (a head that never forgets returns it whole, one that forgets at once returns nothing)."""
    from nanospec_amd.kernels import ops
    from nanospec_amd.parts import retention
    from nanospec_amd.parts.retention import CHUNKS, ChunkPlan

    monkeypatch.setattr(retention, "CHUNKED_FROM", 64)
    n = gap + 1
    decay = torch.tensor([1.0, 0.99, 0.0, 0.9][:H])
    g = torch.Generator().manual_seed(gap)
    q, k, v = torch.zeros(n, H, D), torch.randn(n, H, D, generator=g), torch.randn(n, H, E, generator=g)
    k[:, :, 3] = 0.0
    k[0, :, 3] = 1.0  # only the first token writes channel 3
    q[-1, :, 3] = 1.0  # only the last token reads, and only channel 3
    flat = torch.cat([q.reshape(n, -1), k.reshape(n, -1), v.reshape(n, -1)], dim=1).to(DEV).contiguous()
    want = v[0] * (decay ** gap)[:, None]
    for cuts in ((0, n), tuple(sorted({0, n - 64, n}))):
        state = torch.zeros(3, H * D * E, device=DEV)
        out = torch.empty(n, H * E, device=DEV)
        for a, b in zip(cuts, cuts[1:]):
            ctx = Ctx()
            ctx.requests([b - a], [1], list(range(a, b)), CHUNKS, spare=1)
            if b - a >= 64:
                chunks, rest = ChunkPlan.view(ctx)
                assert rest == 0 and chunks.shape[0] == -(-(b - a) // 64) + 1
                ops.retention_chunks(flat[a:b].contiguous(), decay.to(DEV), state, chunks, ctx.state_slots, H, D, E,
                                     torch.full((chunks.shape[0] * H * D * E,), float("nan"), device=DEV), out[a:b])
            elif b > a:
                ops.retention_scan(flat[a:b].contiguous(), decay.to(DEV), state, ctx.qo_indptr, ctx.state_slots, H, D, E, out=out[a:b])
        assert torch.allclose(out[-1].cpu().view(H, E), want, rtol=1e-4, atol=1e-6), cuts
        assert torch.equal(state[0].cpu(), torch.zeros(H * D * E)) and torch.equal(state[2].cpu(), torch.zeros(H * D * E))


@BOTH
@pytest.mark.parametrize("H,D,R,E,C", [(3, 24, 8, 40, 56), (1, 16, 2, 48, 16), (8, 32, 16, 16, 64), (2, 32, 32, 64, 96), (5, 64, 32, 48, 96), (3, 5, 6, 7, 9)])
def test_latent_attention_with_a_gate_per_channel_over_six_steps(dtype, H, D, R, E, C):
    """The mixer alone over a paged cache whose pages are not in order: a prompt portion, a second one, then single tokens and
    short portions; interleaved rotation, a gate per channel; against the plain mixer over the whole sequence.  One token's
    rotated key part, which no norm bounds, is made so large that it stands out, at a page's first or last place or far back."""
    from nanospec_amd.cache.storage import PagedView
    from nanospec_amd.config import ZipedraConfig
    from nanospec_amd.config.zipedra import ZipedraLayer
    from nanospec_amd.parts import registry

    Wd, T, page = 72, 90, 8
    spec = ZipedraConfig(vocab=8, width=Wd, layers=(), norm_eps=1e-5)._mixer(
        ZipedraLayer(type="latent_attention", heads=H, dim=D, rot_dim=R, vdim=E, kv_rank=C, scale=0.3, rot_base=1000.0))
    part = registry.build("mixer", spec, "m.")
    g = torch.Generator().manual_seed(H * D + R)
    w = {}
    for name, (shape, role) in part.wanted().items():
        w[name] = (torch.randn(shape, generator=g) * (0.15 if role == "linear" else 1.0)).to(dtype)
    assert set(w) == {"m." + n for n in ("q", "dkv", "dkv.norm", "uk", "uv", "g", "o")}
    part.load(lambda name: w[name], dtype, DEV)
    wd = {k: v.double() for k, v in w.items()}
    m = dict(heads=H, dim=D, rot_dim=R, vdim=E, kv_rank=C, scale=0.3, rot={"dims": R, "base": 1000.0})
    pages = -(-T // page)
    order = list(range(pages))
    random.Random(2).shuffle(order)
    for mark in (0, 7, 8, 40):
        x = torch.randn(T, Wd, generator=g).to(dtype)
        plain = lambda y: pz.latent_attention(y.double(), wd, "m.", m, 1e-5, torch.arange(T))
        calm, token = plain(x), x[mark].clone()
        for by in (12.0, -12.0, 24.0, -24.0, 48.0, -48.0):  # (one of the signs meets the last query's favour)
            x[mark] = token * by
            ref = plain(x)
            share = (ref[-1] - calm[-1]).abs().max() / calm[-1].abs().max()
            if share > 0.05:
                break
        assert share > 0.05, "the large key was meant to matter far away"
        cache = PagedView(0, torch.zeros(pages, 1, page, C + R, dtype=dtype, device=DEV), torch.zeros(pages, 1, C, page, dtype=dtype, device=DEV))
        got, at = [], 0
        for n in (37, 30, 1, 1, 2, 19):
            ctx = step_context([n], [at], [order])
            got.append(part.forward(ctx, x[at : at + n].to(DEV), cache, True).cpu())
            at += n
        worst, rms = off(torch.cat(got), ref)
        # (sharp soft-maxes magnify a rounding in single places: the root mean square is what bfloat16 is held to)
        assert worst <= 3e-5 if dtype == torch.float32 else rms <= 0.03, (mark, worst, rms)


@BOTH
@pytest.mark.parametrize("page", [4, 8, 16])
def test_a_key_that_stands_out_at_the_pages_edges(dtype, page):
    """One key/value head with keys and values of two sizes, as a latent layer's cache holds them: all keys small but one,
    placed far back and at a page's first and last place, in a prompt's rows and for a single decoded row, by the kernel that
    the layer runs at these sizes (the matrix cores' in bfloat16)."""
    from nanospec_amd.kernels import ops
    from nanospec_amd.parts.attention import wide_attention

    H, hd, vd, T, scale = 4, 48, 32, 200, 0.3
    g = torch.Generator().manual_seed(page)
    for mark in sorted({0, page - 1, page, 97, T - 2, T - 1, (T // page) * page - 1}):
        keys, vals, q = 0.1 * torch.randn(T, 1, hd, generator=g), torch.randn(T, 1, vd, generator=g), torch.randn(T, H, hd, generator=g)
        keys[mark] = 4.0 * q[T - 1, 0] / scale / hd  # the last query's favourite
        keys, vals, q = keys.to(dtype), vals.to(dtype), q.to(dtype)
        kp, vp, table = paged(keys, vals, page, order_seed=mark)
        s = torch.einsum("thd,jd->htj", q.double(), keys[:, 0].double()) * scale
        s = s.masked_fill(torch.arange(T)[None, None, :] > torch.arange(T)[None, :, None], float("-inf"))
        want = (torch.softmax(s, -1) @ vals[:, 0].double()).transpose(0, 1)
        for first in (0, T - 1):
            n = T - first
            ctx = step_context([n], [first], [table[0].tolist()])
            rows, out = q[first:].reshape(n, H * hd).to(DEV).contiguous(), torch.zeros(n, H * vd, dtype=dtype, device=DEV)
            view = type("V", (), {"k": kp, "v": vp})()
            if ops.wide_attention_takes(dtype, hd, vd, page):
                wide_attention(ctx, rows, out, view, ctx.block_tables[0], H, 1, hd, vd, scale)
            else:
                ops.attention_generic(rows, out, kp, vp, ctx.token_req, ctx.positions, ctx.block_tables[0], H, 1, hd, scale, v_dim=vd)
            err = (out.cpu().double().view(n, H, vd) - want[first:]).abs().max()
            assert err <= (2e-5 if dtype == torch.float32 else 3e-2), (mark, first, float(err))


@BOTH
@pytest.mark.parametrize("W,n,top,ff,shared", [(90, 6, 3, 20, 28), (64, 1, 1, 48, 0), (128, 16, 3, 32, 64), (128, 4, 4, 64, 96), (72, 10, 4, 40, 0)])
@pytest.mark.parametrize("rows", [1, 7, 300])
def test_mixture_of_ungated_experts_through_the_part(dtype, W, n, top, ff, shared, rows):
    """The feed-forward as the framework builds it against the plain one, for one row (streamed experts), a few, and many (the
    sorted, tiled products)."""
    from nanospec_amd.config import ZipedraConfig
    from nanospec_amd.config.zipedra import ZipedraFF
    from nanospec_amd.parts import registry
    from nanospec_amd.weights import random_tensors

    mlp = moe(n, top, ff, shared)
    part = registry.build("ffn", ZipedraConfig(vocab=8, width=W, layers=())._ffn(ZipedraFF.from_hf(mlp)), "")
    tensors = random_tensors(part.wanted(), W + n, torch.float32)
    assert ("shared.sg" in tensors) == bool(shared) and not any(k.endswith("gate") for k in tensors)
    for name, t in tensors.items():
        t *= 30.0 if name == "router" else (10.0 if name.endswith("sg") else 6.0)
    tensors = {k: v.to(dtype) for k, v in tensors.items()}
    part.load(lambda name: tensors[name], dtype, DEV)
    w = {k: v.double() for k, v in tensors.items()}
    x = torch.randn(rows, W, generator=torch.Generator().manual_seed(rows)).to(dtype)
    y = part.forward(Ctx(), x.to(DEV)).cpu().double()
    want = pz.moe(x.double(), w, "", mlp)
    if shared:
        gate = torch.sigmoid(x.double() @ w["shared.sg"][0])
        assert rows == 1 or gate.max() - gate.min() > 0.3, "the shared expert's gate was meant to vary"
    if dtype == torch.float32:
        assert (y - want).abs().max() <= 1e-4 * want.abs().max()
    else:  # (a row whose router scores lie within rounding of each other may take another expert)
        err = (y - want).pow(2).mean(-1).sqrt() / want.pow(2).mean().sqrt()
        assert (err > 0.05).sum() <= max(1, rows // 25), err.max()


@pytest.mark.parametrize("rows", [1, 3, 20])
def test_router_leaves_the_rows_that_belong_to_no_expert_alone(rows):
    """Two rows below the experts': their logits come back behind the experts', they are never chosen however large they are, and
    the weights are the chosen experts' soft-max scores over their sum."""
    from nanospec_amd.kernels import ops

    n, top, W, extra = 9, 3, 40, 2
    g = torch.Generator().manual_seed(rows)
    h, router = torch.randn(rows, W, generator=g), torch.randn(n + extra, W, generator=g)
    router[n:] *= 10.0
    sel, wt = torch.empty(rows, top, dtype=torch.int32, device=DEV), torch.empty(rows, top, device=DEV)
    z = torch.empty(rows, n + extra, device=DEV)
    ops.moe_route(h.to(DEV), router.to(DEV), None, top, sel, wt, logits=z, extra=extra)
    want_sel, want_wt = pz.route(h, {"router": router[:n]}, "", {"top": top})
    assert sel.cpu().tolist() == want_sel.tolist()
    assert torch.allclose(wt.cpu(), want_wt, rtol=1e-5) and torch.allclose(z.cpu(), h @ router.T, rtol=1e-4, atol=1e-3)


@BOTH
@pytest.mark.parametrize("W", [64, 90, 4100])
@pytest.mark.parametrize("S", [1, 2])
def test_two_outputs_are_written_into_the_stream_at_once(dtype, W, S):
    """x_t <- sum_s mix[s, t] x_s + gain[t] (y + y2) in 32-bit and the normed read behind it; with a bias and a norm behind the
    sum as well; with a write alone."""
    from nanospec_amd.kernels import ops

    n, eps = 7, 1e-4
    g = torch.Generator().manual_seed(W)
    x, mix, gain, coeff = (torch.randn(s, generator=g) for s in ((n, S, W), (S, S), (S,), (S,)))
    y, y2, wn, b, wb = (torch.randn(s, generator=g).to(dtype) for s in ((n, W), (n, W), (W,), (W,), (W,)))
    d = lambda t: t.to(DEV)
    for post in (None, ops.PostNorm(bias=d(b)), ops.PostNorm(d(b), d(wb), eps, 0.0)):
        total = y.double() + y2.double()
        if post is not None:
            total = total + b.double()
            if post.weight is not None:
                total = pz.rms(total, eps) * wb.double()
        new = torch.einsum("nsw,st->ntw", x.double(), mix.double()) + gain.double()[None, :, None] * total[:, None, :]
        xs = d(x).clone()
        out = ops.stream_step(xs, ops.PendingWrite(d(y), d(mix), d(gain), post, d(y2)), d(coeff), d(wn), eps)
        assert torch.allclose(xs.cpu().double(), new, atol=2e-5, rtol=1e-5)
        u = (new * coeff.double()[None, :, None]).sum(1)
        want = pz.rms(u, eps) * wn.double()
        assert (out.cpu().double() - want).abs().max() <= (1e-4 if dtype == torch.float32 else 2e-2) * want.abs().max()
        xs = d(x).clone()
        assert ops.stream_step(xs, ops.PendingWrite(d(y), d(mix), d(gain), post, d(y2))) is None
        assert torch.allclose(xs.cpu().double(), new, atol=2e-5, rtol=1e-5)


@BOTH
@pytest.mark.parametrize("W", [64, 90, 4100])
def test_a_read_followed_by_a_table_row(dtype, W):
    """[stream after the pending write | scale * table row of the token], the stream itself left as it was where the caller says
    that nobody reads it again (in the one-pass kernel)."""
    from nanospec_amd.kernels import ops

    n = 6
    g = torch.Generator().manual_seed(W)
    x, y, table = torch.randn(n, 1, W, generator=g), torch.randn(n, W, generator=g).to(dtype), torch.randn(20, W, generator=g).to(dtype)
    ids = torch.tensor([3, 19, 0, 3, 7, 8], dtype=torch.int32)
    one = torch.ones(1, device=DEV)
    for pending in (None, ops.PendingWrite(y.to(DEV), torch.ones(1, 1, device=DEV), one)):
        xs = x.to(DEV)
        out = ops.stream_step(xs, pending, one, None, 0.0, store=False, dtype=dtype, tail=(table.to(DEV), ids.to(DEV), 0.5))
        want = torch.cat([x[:, 0] + (y.float() if pending is not None else 0.0), table.float()[ids.long()] * 0.5], dim=1).to(dtype)
        assert out.shape == (n, 2 * W) and torch.allclose(out.cpu().float(), want.float(), rtol=1e-2 if dtype == torch.bfloat16 else 1e-6, atol=1e-6)
    with pytest.raises(ops.KernelRefused):
        ops.stream_step(x.to(DEV), None, one, None, 0.0, dtype=dtype, tail=(table.to(DEV), ids.to(DEV)[:3], 0.5))


@BOTH
@pytest.mark.parametrize("width", [40, 512, 1000, 2048])
def test_the_norm_over_all_heads_with_a_sigmoid_gate(dtype, width):
    from nanospec_amd.kernels import ops

    n = 5
    g = torch.Generator().manual_seed(width)
    o, wn = 5.0 * torch.randn(n, width, generator=g), 1.0 + 0.3 * torch.randn(width, generator=g)
    gate = (2.0 * torch.randn(n, width + 8, generator=g)).to(dtype)
    out = ops.gated_rms(o.to(DEV), gate.to(DEV)[:, 8:], wn.to(DEV), 1e-5, 1, out=torch.empty(n, width, dtype=dtype, device=DEV))
    want = pz.rms(o.double(), 1e-5) * wn.double() * torch.sigmoid(gate[:, 8:].double())
    worst, _ = off(out, want)
    assert worst <= (1e-5 if dtype == torch.float32 else 8e-3)


@BOTH
@pytest.mark.parametrize("rows", [1, 5, 40])
def test_the_squared_relu_behind_a_product(dtype, rows):
    """In the streaming product's epilogue for few rows, a kernel of its own otherwise: the same values either way."""
    from nanospec_amd.kernels import ops
    from nanospec_amd.parts.linear import LinearWeight

    g = torch.Generator().manual_seed(rows)
    w, x = torch.randn(72, 128, generator=g).to(dtype), torch.randn(rows, 128, generator=g).to(dtype)
    got = LinearWeight(w.to(DEV))(x.to(DEV), act="relu2")
    want = pz.relu2(x.double() @ w.double().T)
    worst, _ = off(got, want)
    assert (want == 0).any() and worst <= (1e-5 if dtype == torch.float32 else 1.5e-2)
    z = torch.randn(rows, 33, generator=g).to(dtype)
    worst, _ = off(ops.activation(z.to(DEV), "relu2"), pz.relu2(z.double()))
    assert worst <= (1e-6 if dtype == torch.float32 else 4e-3)
