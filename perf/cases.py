"""The work that is timed to judge a change: whole calls of the engine, made the way a program of its users makes them.

Two kinds of model are run.  "quant" cases load a GGUF file of the shapes and quantised types the engine serves (a whole TinyLlama-1.1B as the draft, a few layers of Llama-2-7B and Llama-2-70B with
the full output head as the target: the cost of a call is additive per layer); "folder" cases load a described folder (config.json + model.safetensors) of three designs that between them hold the
latent, windowed, chunked and differential attentions, the three recurrences, dense and routed feed-forwards.  All weights are synthetic.

A pass is what one request of such a program costs: a token, a verify batch, a prompt, a prompt followed by given tokens, or several continuations of a shared prefix.  It leaves the context as it
found it (the tokens it added are taken back), so it can be repeated.
"""
import ctypes
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from pipeinfer_amd import lib as L
from pipeinfer_amd import llama as LL
from pipeinfer_amd.tools import gguf as G
from pipeinfer_amd.tools import synth
from pipeinfer_amd.tools.hybrid_bench import SIZES, VIKARAX, rerizen_ff

WEIGHTS_SEED = 0x5EED        # every state of a case runs the same model; tokens come from the state's seed


def listed():
    return [
        # one token of the draft model: 22 small layers, the call that gates speculation
        {"name": "draft token", "kind": "quant", "model": "tinyllama-1.1b", "type": "q4_k_m", "first": 0, "layers": 22, "past": 200, "tokens": 1, "branches": 1, "score": True},
        # one token of the target: weights streamed from memory once
        {"name": "target token", "kind": "quant", "model": "llama-2-70b", "type": "q4_k_m", "first": 11, "layers": 2, "past": 250, "tokens": 1, "branches": 1, "score": True},
        # the verify batch of a speculation tree with three branches
        {"name": "target verify 7", "kind": "quant", "model": "llama-2-70b", "type": "q4_k_m", "first": 11, "layers": 2, "past": 250, "tokens": 7, "branches": 3, "score": True},
        # the benchmark's prompt
        {"name": "target prompt 128", "kind": "quant", "model": "llama-2-70b", "type": "q4_k_m", "first": 11, "layers": 2, "past": 0, "tokens": 128, "branches": 1, "score": False},
        # a longer, ragged prompt of a model in the older 32-value block type
        {"name": "7b q4_0 prompt 333", "kind": "quant", "model": "llama-2-7b", "type": "q4_0", "first": 4, "layers": 4, "past": 0, "tokens": 333, "branches": 1, "score": False},
        # a short request to a small folder model: a prompt of a sentence and eight tokens behind it
        {"name": "fasovik request", "kind": "folder", "design": "Fasovik", "size": "w1024", "past": 0, "sequences": 1, "prompt": 24, "steps": 8, "score": False},
        # a prompt of the usual pass length through latent attention, lightning layers and routed experts
        {"name": "fasovik prompt 512", "kind": "folder", "design": "Fasovik", "size": "w2048", "past": 0, "sequences": 1, "prompt": 512, "steps": 0, "score": False},
        # the largest: a document in one pass
        {"name": "fasovik prompt 2048", "kind": "folder", "design": "Fasovik", "size": "w4096", "past": 0, "sequences": 1, "prompt": 2048, "steps": 0, "score": False},
        # four continuations sampled from one shared conversation
        {"name": "letevik continuations", "kind": "folder", "design": "Letevik", "size": "w2048", "past": 700, "sequences": 4, "prompt": 0, "steps": 8, "score": False},
        # a ragged prompt longer than the attention window
        {"name": "letevik prompt 1000", "kind": "folder", "design": "Letevik", "size": "w2048", "past": 0, "sequences": 1, "prompt": 1000, "steps": 0, "score": False},
        # a text scored token by token: every logit is wanted
        {"name": "rafusun score 333", "kind": "folder", "design": "Rafusun", "size": "w2048", "past": 0, "sequences": 1, "prompt": 333, "steps": 0, "score": True},
        # eight users served together: short prompts in one pass, then a token each per pass
        {"name": "rafusun batch of 8", "kind": "folder", "design": "Rafusun", "size": "w4096", "past": 0, "sequences": 8, "prompt": 37, "steps": 8, "score": False},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.4:
        model, types, first, layers = rng.choice([("tinyllama-1.1b", ("q4_k_m", "q5_k_m", "q4_0"), 0, 22), ("llama-2-7b", ("q4_0", "q4_k_m"), 4, 4), ("llama-2-70b", ("q4_k_m", "q5_k_m"), 11, 2)])
        case = {"kind": "quant", "model": model, "type": rng.choice(types), "first": first, "layers": layers}
        what = rng.choice(("token", "verify", "prompt"))
        if what == "prompt":
            case.update(past=0, tokens=_log_uniform(rng, 9, 300), branches=1, score=rng.random() < 0.3)
        else:
            case.update(past=_log_uniform(rng, 30, 900), tokens=1 if what == "token" else rng.randint(2, 8), branches=1 if what == "token" else rng.randint(1, 3), score=True)
        return case
    case = {"kind": "folder", "design": rng.choice(("Fasovik", "Letevik", "Rafusun")), "size": rng.choice(("w1024", "w2048", "w4096"))}
    what = rng.choice(("request", "prompt", "continuations", "batch"))
    if what == "request":
        case.update(past=0, sequences=1, prompt=_log_uniform(rng, 5, 200), steps=rng.randint(2, 12), score=False)
    elif what == "prompt":
        case.update(past=0, sequences=1, prompt=_log_uniform(rng, 60, 1500), steps=0, score=False)
        case["score"] = case["prompt"] <= 400 and rng.random() < 0.4
    elif what == "continuations":
        case.update(past=_log_uniform(rng, 100, 1200), sequences=rng.randint(1, 8), prompt=rng.choice((0, rng.randint(1, 40))), steps=rng.randint(2, 8), score=False)
    else:
        case.update(past=0, sequences=rng.randint(2, 12), prompt=rng.randint(8, 60), steps=rng.randint(2, 8), score=False)
    return case


# ---- models --------------------------------------------------------------------------------------------------------------------------------
def _quant_file(case, folder):
    path = os.path.join(folder, "model.gguf")
    synth.write_model(path, case["model"], case["type"], seed=WEIGHTS_SEED, layers=(case["first"], case["layers"]))
    return path


def _folder_plan(case):
    """(config, {tensor: (shape, fill)}) of a design at one of the repository's sizes"""
    design, size = case["design"], case["size"]
    width, n_layer, heads, dim, vdim, rank, n_exp, n_id, top, ff, vocab = SIZES[size]
    kv_heads, rot, chunk, r_heads, r_dim = VIKARAX[size][:5]
    hd, hv, mat = heads * dim, heads * vdim, lambda *shape: (shape, "matrix")
    gain, bias = lambda *shape: (shape, "gain"), lambda *shape: (shape, "bias")
    pair = {"buckets": 65536, "mul_prev": 8191, "mul_cur": 31}
    T, layers = {"embed": mat(vocab, width), "final.norm": gain(width)}, []
    cfg = {"architecture": design, "vocab": vocab, "width": width, "norm": {"eps": 1e-5}, "layers": layers}
    if design == "Fasovik":
        cfg.update(embedding={"scale": 1.0}, residual_mult=0.5)
        T["embed"], T["final.norm"] = ((vocab, width), "routed embedding"), bias(width)
    elif design == "Rafusun":
        cfg.update(embedding={"scale": 1.0, "bigram": pair}, postln_alpha=2.0)
        T.update({"embed": ((vocab, width), "embedding"), "bigram": ((65537, width), "embedding"), "head": mat(vocab, width)})
    else:
        cfg.update(embedding={"bigram": pair}, loop={"start": 1, "stop": min(3, n_layer), "times": 1})
        T.update({"bigram": ((65537, width), "embedding"), "loop.step": ((1, width), "bias"), "embed": ((vocab, width), "embedding")})
    for i in range(n_layer):
        p, q = "l%d." % i, "l%d.mix." % i
        if design == "Fasovik":
            T.update({p + "norm1": bias(width), p + "norm2": bias(width), q + "q": mat(hd, width), q + "o": mat(width, hv)})
            if i % 2:
                kind, mx = "lightning", {"heads": heads, "dim": dim, "vdim": vdim, "decay": [float(1.0 - 2.0 ** (-3 - 5 * h / heads)) for h in range(heads)]}
                T.update({q + "k": mat(hd, width), q + "v": mat(hv, width), q + "g": mat(hv, width), q + "norm": gain(hv)})
            else:
                kind, mx = "latent_attention", {"heads": heads, "dim": dim, "vdim": vdim, "kv_rank": rank, "scale": dim ** -0.5}
                T.update({q + "dkv": mat(rank, width), q + "dkv.norm": gain(rank), q + "uk": mat(hd, rank), q + "uv": mat(hv, rank), q + "sink": bias(heads)})
            mlp = {"kind": "moe", "expert": {"ff": ff}, "router": {"experts": n_exp, "identity": n_id, "top": top}}
            T.update({p + "mlp.router": ((n_exp + n_id, width), "router"), p + "mlp.correction": ((n_exp + n_id,), "small")})
            for e in range(n_exp):
                T.update({p + "mlp.e%d.up" % e: mat(ff, width), p + "mlp.e%d.down" % e: mat(width, ff)})
        elif design == "Rafusun":
            T.update({p + "norm1": gain(width), p + "ls1": gain(width)})
            if i % 2 == 0:
                kind, mx, mlp = "channel_delta", {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim, "conv": 4}, None
                for n, rows in (("q", kv_heads * dim), ("k", kv_heads * dim), ("v", hv)):
                    T.update({q + n: mat(rows, width), q + n + ".conv": ((rows, 4), "taps")})
                T.update({q + "b": mat(heads, width), q + "A_log": bias(heads), q + "dt_bias": ((hd,), "low"), q + "a1": mat(64, width), q + "a2": mat(hd, 64), q + "g1": mat(64, width), q + "g2": mat(hv, 64),
                          q + "norm": gain(vdim), q + "o": mat(width, hv)})
            else:
                inner = r_heads * r_dim
                kind, mlp = "parallel", {"kind": "dense", "ff": 4 * ff}
                left = {"heads": heads, "kv_heads": kv_heads, "dim": dim, "vdim": vdim, "scale": dim ** -0.5, "softcap": 30.0, "rot": {"dims": rot, "base": 10000.0}, "mask": {"size": chunk}}
                mx = {"left": left, "right": {"heads": r_heads, "dim": r_dim}}
                T.update({q + "left.q": mat(hd, width), q + "left.k": mat(kv_heads * dim, width), q + "left.v": mat(kv_heads * vdim, width), q + "left.o": mat(width, hv), q + "left.out": gain(width)})
                T.update({q + "right.mu." + n: ((width,), "unit") for n in "rkvgw"})
                T.update({q + "right." + n: mat(inner, width) for n in "rkvg"})
                T.update({q + "right.w1": mat(64, width), q + "right.w2": mat(inner, 64), q + "right.w0": ((inner,), "low"), q + "right.u": bias(r_heads, r_dim), q + "right.norm": gain(inner),
                          q + "right.o": mat(width, inner), q + "right.out": gain(width)})
                T.update({p + "norm2": gain(width), p + "ls2": gain(width), p + "mlp.gate": mat(4 * ff, width), p + "mlp.up": mat(4 * ff, width), p + "mlp.down": mat(width, 4 * ff)})
        else:
            if i % 2:
                kind = "attention"
                mx = {"heads": heads, "kv_heads": kv_heads, "dim": dim // 2, "vdim": vdim, "scale": (dim // 2) ** -0.5, "diff": 0.4, "conv": 4, "rot": {"dims": dim // 2, "base": 10000.0},
                      "mask": {"size": chunk, "keep_first": 4}}
                for n, rows in (("q", hd), ("k", kv_heads * dim), ("v", kv_heads * vdim)):
                    T.update({q + n: mat(rows, width), q + n + ".conv": ((rows, 4), "taps")})
                T.update({q + n: bias(dim // 2) for n in ("lq1", "lk1", "lq2", "lk2")})
            else:
                kind, q_rank, r = "latent_attention", width // 2, dim // 2
                mx = {"heads": heads, "dim": dim, "rot_dim": r, "vdim": vdim, "q_rank": q_rank, "kv_rank": rank, "scale": (dim + r) ** -0.5, "rot": {"dims": r, "base": 10000.0}}
                T.update({q + "dq": mat(q_rank, width), q + "dq.norm": gain(q_rank), q + "uq": mat(heads * (dim + r), q_rank), q + "dkv": mat(rank + r, width), q + "dkv.norm": gain(rank),
                          q + "uk": mat(hd, rank), q + "uv": mat(hv, rank), q + "sink": bias(heads), q + "g": mat(hv, width)})
            f = rerizen_ff(size)
            mlp = {"kind": "dense", "ff": f, "limit": 7.0}
            T.update({q + "o": mat(width, hv), p + "norm1": gain(width), p + "norm2": gain(width), p + "mlp.gate": mat(f, width), p + "mlp.up": mat(f, width), p + "mlp.down": mat(width, f)})
        layers.append({"type": kind, "mixer": mx, "mlp": mlp})
    return cfg, T


def _folder_tensors(case):
    """the model's bfloat16 tensors, on the GPU.  The router's rows are directions that a token's embedding has a large share of, two for each token: which experts a token takes is as decided as in
    a trained router, and no rounding moves it"""
    cfg, plan = _folder_plan(case)
    gen = torch.Generator(device="cuda").manual_seed(WEIGHTS_SEED)

    def normal(shape):
        return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)
    tensors, directions = {}, None
    n_out = max([t[0][0] for t in plan.values() if t[1] == "router"], default=0)
    if n_out:
        directions = torch.nn.functional.normalize(normal((n_out, cfg["width"])), dim=1)
    for name, (shape, fill) in plan.items():
        if fill == "matrix":
            t = normal(shape) * shape[-1] ** -0.5
        elif fill == "embedding":
            t = normal(shape) * 0.7
        elif fill == "routed embedding":
            tok = torch.arange(shape[0], device="cuda")
            a = tok % n_out
            b = (a + 1 + tok // n_out % (n_out - 1)) % n_out
            t = normal(shape) + 0.3 * cfg["width"] ** 0.5 * (directions[a] + 0.9 * directions[b])
        elif fill == "router":
            t = directions + 0.1 * normal(shape) * shape[-1] ** -0.5
        elif fill == "gain":
            t = 1.0 + 0.1 * normal(shape)
        elif fill == "taps":
            t = 0.3 * normal(shape)
            t[:, -1] += 1.0
        elif fill == "unit":
            t = torch.rand(shape, generator=gen, device="cuda")
        elif fill == "low":
            t = normal(shape) - 1.5
        else:
            t = normal(shape) * (0.01 if fill == "small" else 0.1)
        tensors[name] = t.to(torch.bfloat16)
    return cfg, tensors


def _folder_file(case, folder):
    import json
    import struct
    cfg, tensors = _folder_tensors(case)
    head, at = {}, 0
    for name, t in tensors.items():
        head[name] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + 2 * t.numel()]}
        at += 2 * t.numel()
    text = json.dumps(head).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(folder, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)) + text)
        for t in tensors.values():
            t.contiguous().view(torch.int16).cpu().numpy().tofile(f)
    with open(os.path.join(folder, "config.json"), "w") as f:
        json.dump(cfg, f)
    return folder


def _model_key(case):
    return tuple(case[k] for k in (("model", "type", "first", "layers") if case["kind"] == "quant" else ("design", "size")))


_models = {}        # a program loads a model once and opens contexts on it


def _model(case):
    key = _model_key(case)
    if key not in _models:
        folder = tempfile.mkdtemp(prefix="perf_model_")
        try:
            _models[key] = LL.Model((_quant_file if case["kind"] == "quant" else _folder_file)(case, folder))
        finally:
            shutil.rmtree(folder)        # (the loader keeps the file mapped)
    return _models[key]


# ---- inputs --------------------------------------------------------------------------------------------------------------------------------
def _tokens(case, seed):
    """quant: {"past": [past], "batch": (tokens, positions, sequence lists)}; folder: {"past": [past], "own": [sequences][prompt + steps]}"""
    rng = np.random.default_rng([seed, 7])
    vocab = SIZES[case["size"]][10] if case["kind"] == "folder" else synth.SPECS[case["model"]][6]
    past = rng.integers(3, vocab, case["past"])
    if case["kind"] == "folder":
        return {"past": past, "own": rng.integers(3, vocab, (case["sequences"], case["prompt"] + case["steps"]))}
    n, nb = case["tokens"], case["branches"]
    toks = rng.integers(3, vocab, n)
    if nb == 1:
        return {"past": past, "batch": (toks, case["past"] + np.arange(n), [[0]] * n)}
    # the accepted token belongs to every branch, the drafted ones to a branch each, round the branches
    return {"past": past, "batch": (toks, np.array([case["past"] + (0 if i == 0 else 1 + (i - 1) // nb) for i in range(n)]), [list(range(nb)) if i == 0 else [(i - 1) % nb] for i in range(n)])}


class State:
    def __init__(self, case, seed):
        self.case, self.tokens = case, _tokens(case, seed)
        model = _model(case)
        past = [int(t) for t in self.tokens["past"]]
        if case["kind"] == "quant":
            width = case["tokens"]
            self.ctx = LL.Context(model, n_ctx=(case["past"] + case["tokens"] + 127) // 64 * 64, n_batch=max(128, width))
            toks, pos, seqs = self.tokens["batch"]
            self.prompt = LL.Batch(toks, pos, seqs)
        else:
            b, width, steps = case["sequences"], case["sequences"] * case["prompt"], case["steps"]
            self.ctx = LL.Context(model, n_ctx=(case["past"] + b * (case["prompt"] + steps) + 127) // 64 * 64, n_batch=max(512, width))
            self.ctx.set_precision(False)
            self.ctx.set_state_slots(b + 1)
            own, p0, at = self.tokens["own"], case["past"], case["prompt"]
            self.prompt = LL.Batch(own[:, :at].reshape(-1), np.tile(p0 + np.arange(at), b), [[1 + s] for s in range(b) for _ in range(at)]) if at else None
            self.steps = [([int(t) for t in own[:, at + k]], [p0 + at + k] * b, [[1 + s] for s in range(b)]) for k in range(steps)]
        if self.prompt and not case["score"]:        # a prompt's caller wants what follows its last token
            last = len(self.prompt.tok) // case.get("sequences", 1)
            self.prompt.lg[:] = 0
            self.prompt.lg[last - 1::last] = 1
        self.ctx.prepare()
        if past:
            self.ctx.feed(past, 0)
            for s in range(1, case.get("branches", 1)):
                self.ctx.seq_cp(0, s, -1, -1)
        self.rows = None if not self.prompt else np.flatnonzero(self.prompt.lg)

    def __del__(self):
        if getattr(self, "ctx", None) is not None:
            self.ctx.free()


def prepare(case, seed):
    return State(case, seed)


def _prompt(state):
    """one pass over the prompt's batch; the logits that were asked for"""
    ctx, n = state.ctx, len(state.prompt.tok)
    if ctx.lib.llama_decode(ctx.h, state.prompt.c) != 0:
        raise RuntimeError("llama_decode: " + ctx.lib.pipeinfer_context_error(ctx.h).decode())
    buf = ctypes.cast(ctx.lib.llama_get_logits(ctx.h), ctypes.POINTER(ctypes.c_float * (n * ctx.n_vocab))).contents        # the context's own buffer,
    buf.owner = state                                                                                                          # which lives as long as what is returned
    logits = np.ctypeslib.as_array(buf).reshape(n, ctx.n_vocab)
    return logits if len(state.rows) == n else logits[state.rows]


def run(state):
    case, ctx = state.case, state.ctx
    if case["kind"] == "quant":
        if case["past"]:
            ctx.seq_rm(-1, case["past"], -1)        # what the pass before this one added
        else:
            ctx.kv_clear()
        return _prompt(state)
    out = []
    if case["past"]:
        for s in range(case["sequences"]):
            ctx.seq_cp(0, 1 + s, -1, -1)
    else:
        ctx.kv_clear()
    if state.prompt:
        got = _prompt(state)
        out.append(got.copy() if state.steps else got)
    for tokens, pos, seqs in state.steps:
        out.append(ctx.decode(tokens, pos, seqs))
    if case["past"]:
        for s in range(case["sequences"]):
            ctx.seq_rm(1 + s, -1, -1)
    return out


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------------------------
def work(case):
    if case["kind"] == "quant":
        _, _, n_embd, n_head, n_kv, _, vocab, _ = synth.SPECS[case["model"]]
        plan = [t for t in synth.tensor_plan(case["model"], case["type"], layers=(case["first"], case["layers"])) if t[0] != "token_embd.weight"]
        n, cells = case["tokens"], case["past"] + case["tokens"]
        rows = n if case["score"] else 1
        params = sum(ne[0] * ne[1] for name, ne, _, _ in plan if len(ne) == 2 and name != "output.weight")
        kv = 4 * n_embd * n_kv // n_head * case["layers"]
        seen = n * case["past"] + n * (n + 1) // 2
        return {"bytes": sum(G.nbytes(t, ne) for _, ne, t, _ in plan) + kv * cells + 4 * vocab * rows, "flops": 2 * params * n + 2 * n_embd * vocab * rows + 4 * n_embd * case["layers"] * seen}
    cfg, plan = _folder_plan(case)
    heads, dim, vdim, rank = SIZES[case["size"]][2:6]
    tied = "head" not in plan
    total = {"bytes": 0, "flops": 0}

    def one_pass(sequences, tokens, past, rows):
        n = sequences * tokens
        for name, (shape, _) in plan.items():
            if len(shape) != 2 or name in ("bigram", "loop.step") or name.endswith(".conv"):
                continue
            size = shape[0] * shape[1]
            if name == "head" or name == "embed":
                if name == "head" or tied:
                    total["bytes"] += 2 * size
                    total["flops"] += 2 * size * rows
                continue
            share = 1.0
            if ".mlp.e" in name:
                r = cfg["layers"][0]["mlp"]["router"]
                share = r["top"] / (r["experts"] + r["identity"])
                total["bytes"] += 2 * size * min(1.0, share * n)
            else:
                total["bytes"] += 2 * size
            total["flops"] += 2 * size * n * share
        seen = sequences * (tokens * past + tokens * (tokens + 1) // 2)
        for layer in cfg["layers"]:
            mx = layer["mixer"].get("left", layer["mixer"])
            window = (mx.get("mask") or {}).get("size")
            pairs = min(seen, n * window) if window else seen
            if layer["type"] == "latent_attention":
                r = mx.get("rot_dim", 0)
                total["flops"] += 2 * heads * (dim + r + vdim) * pairs
                total["bytes"] += 4 * (rank + r) * (past + n)
            elif layer["type"] in ("attention", "parallel"):
                total["flops"] += (2 if layer["type"] == "parallel" else 4) * heads * (mx["dim"] + vdim) * pairs
                total["bytes"] += 4 * mx["kv_heads"] * (mx["dim"] * (1 if layer["type"] == "parallel" else 2) + vdim) * (min(past, window) + n)
            if layer["type"] in ("lightning", "channel_delta"):
                total["flops"] += (4 if layer["type"] == "lightning" else 8) * heads * dim * vdim * n
                total["bytes"] += 8 * heads * dim * vdim * sequences
            if layer["type"] == "parallel":
                r = layer["mixer"]["right"]
                total["flops"] += 4 * r["heads"] * r["dim"] ** 2 * n
                total["bytes"] += 8 * r["heads"] * r["dim"] ** 2 * sequences
        total["bytes"] += 4 * SIZES[case["size"]][10] * rows

    b, n = case["sequences"], case["prompt"]
    if n:
        one_pass(b, n, case["past"], b * n if case["score"] else b)
    for k in range(case["steps"]):
        one_pass(b, 1, case["past"] + n + k, b)
    return total


def tolerance(case):
    # a quantised model's logits are defined to the bit (sums in the order of the file format's reference arithmetic)
    if case["kind"] == "quant":
        return "exact"
    # bfloat16 matrix inputs, everything else in 32 bits: four times the distance from the same in 64 bits
    return {"rel": {"Fasovik": 0.01, "Rafusun": 0.0125, "Letevik": 0.017}[case["design"]]}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------------------------
def _half(raw):
    return raw.contiguous().view(torch.float16).to(torch.float64)


def _scales_and_mins(s):
    """the eight 6-bit scales and mins of twelve bytes"""
    s = s.to(torch.int32)
    lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
    return torch.cat([lo & 63, (hi & 15) | (lo >> 6) << 4], 1).double(), torch.cat([mid & 63, (hi >> 4) | (mid >> 6) << 4], 1).double()


def _dequantised(kind, ne, raw):
    """the matrix [rows][columns] in float64, on the GPU"""
    b = torch.from_numpy(np.array(raw)).cuda()
    if kind == G.T_F32:
        return b.view(torch.float32).double().reshape(tuple(reversed(ne)))
    if kind == G.T_Q4_0:
        b = b.view(-1, 18)
        q = b[:, 2:]
        x = _half(b[:, :2]) * (torch.cat([q & 15, q >> 4], 1).double() - 8)
    elif kind in (G.T_Q4_K, G.T_Q5_K):
        b = b.view(-1, G.TSIZE[kind])
        sc, mn = _scales_and_mins(b[:, 4:16])
        q = b[:, -128:].reshape(-1, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32)
        if kind == G.T_Q5_K:
            bit = torch.arange(8, device="cuda", dtype=torch.uint8).view(1, 8, 1)
            q = q + (((b[:, None, 16:48] >> bit) & 1) << 4)
        x = (_half(b[:, 0:2]) * sc)[:, :, None] * q.double() - (_half(b[:, 2:4]) * mn)[:, :, None]
    elif kind == G.T_Q6_K:
        b = b.view(-1, 210)
        lo, hi = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 1, 32)
        q = torch.cat([lo & 15, lo >> 4], 2) | ((torch.cat([hi, hi >> 2, hi >> 4, hi >> 6], 2) & 3) << 4)
        x = (_half(b[:, 208:210]) * b[:, 192:208].contiguous().view(torch.int8).double())[:, :, None] * (q.reshape(-1, 16, 16).double() - 32)
    else:
        raise ValueError(kind)
    return x.reshape(ne[1], ne[0])


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, pos, dims, base, neighbours):
    """the first `dims` values of the last axis turned in pairs by pos * base^(-2i/dims); x [..., tokens, heads, values], pos [tokens]"""
    a = pos[:, None].double() * base ** (-2.0 * torch.arange(dims // 2, device=x.device, dtype=torch.float64) / dims)
    c, s = a.cos()[:, None], a.sin()[:, None]
    first, second = (slice(0, dims, 2), slice(1, dims, 2)) if neighbours else (slice(0, dims // 2), slice(dims // 2, dims))
    out = x.clone()
    out[..., first], out[..., second] = x[..., first] * c - x[..., second] * s, x[..., second] * c + x[..., first] * s
    return out


def _exact_quant(case, seed):
    _, _, n_embd, n_head, n_kv, _, vocab, _ = synth.SPECS[case["model"]]
    folder = tempfile.mkdtemp(prefix="perf_model_")
    try:
        _, tensors = G.read_gguf(_quant_file(case, folder))
    finally:
        shutil.rmtree(folder)

    def weight(name):
        ne, kind, raw = tensors[name]
        return _dequantised(kind, ne, raw)
    t = _tokens(case, seed)
    toks, pos, seqs = t["batch"]
    past, n, hd = case["past"], case["tokens"], n_embd // n_head
    everyone = list(range(case["branches"]))
    pos = torch.tensor(np.concatenate([np.arange(past), pos]), device="cuda")
    of = [everyone] * past + list(seqs)
    shares = torch.tensor([[len(set(a) & set(b)) > 0 for b in of] for a in of[past:]], device="cuda")
    sees = torch.ones(past + n, past + n, dtype=torch.bool, device="cuda")
    sees[past:] = shares
    sees &= pos[None, :] <= pos[:, None]
    ne, kind, raw = tensors["token_embd.weight"]
    row = G.nbytes(kind, (ne[0],))
    ids = np.concatenate([t["past"], toks]).astype(np.int64)
    x = _dequantised(kind, (ne[0], len(ids)), np.concatenate([raw[i * row:(i + 1) * row] for i in ids]))
    for i in range(case["layers"]):
        p = "blk.%d." % i
        h = _rms(x, 1e-5) * weight(p + "attn_norm.weight")
        q, k, v = (h @ weight(p + "attn_%s.weight" % c).T for c in "qkv")
        q = _turn(q.view(-1, n_head, hd), pos, hd, 10000.0, True)
        k = _turn(k.view(-1, n_kv, hd), pos, hd, 10000.0, True).repeat_interleave(n_head // n_kv, 1)
        v = v.view(-1, n_kv, hd).repeat_interleave(n_head // n_kv, 1)
        s = q.transpose(0, 1) @ k.permute(1, 2, 0) * hd ** -0.5
        a = torch.softmax(s.masked_fill(~sees, -math.inf), -1) @ v.transpose(0, 1)
        x = x + a.transpose(0, 1).reshape(-1, n_embd) @ weight(p + "attn_output.weight").T
        h = _rms(x, 1e-5) * weight(p + "ffn_norm.weight")
        x = x + (torch.nn.functional.silu(h @ weight(p + "ffn_gate.weight").T) * (h @ weight(p + "ffn_up.weight").T)) @ weight(p + "ffn_down.weight").T
    x = x[past:] if case["score"] else x[-1:]
    return ((_rms(x, 1e-5) * weight("output_norm.weight")) @ weight("output.weight").T).cpu().numpy()


def _conv(w, x):
    """a causal convolution per channel over x [sequences][tokens][channels]; the last tap weighs the token itself"""
    taps, n = w.shape[1], x.shape[1]
    padded = torch.nn.functional.pad(x, (0, 0, taps - 1, 0))
    return sum(padded[:, k:k + n] * w[:, k] for k in range(taps))


def _softmax_with(s, sink):
    """soft-max over the last axis with one more term e^sink in the denominator"""
    top = torch.maximum(s.amax(-1, keepdim=True), sink)
    e = torch.exp(s - top)
    return e / (e.sum(-1, keepdim=True) + torch.exp(sink - top))


def _exact_folder(case, seed):
    cfg, tensors = _folder_tensors(case)
    T = {}

    def w(name):
        if name not in T:
            T[name] = tensors[name].double()
        return T[name]
    tok = _tokens(case, seed)
    b, eps = case["sequences"], cfg["norm"]["eps"]
    ids = torch.tensor(np.concatenate([np.tile(tok["past"], (b, 1)), tok["own"]], 1), device="cuda").long()        # [sequences][tokens]
    n = ids.shape[1]
    pos = torch.arange(n, device="cuda")
    causal = pos[None, :] <= pos[:, None]
    heads, dim, vdim = SIZES[case["size"]][2:5]

    def split(x, h):
        return x.view(b, n, h, -1)

    def attend(p, v):        # weights [b][heads][n][n] over values [b][n][heads][vdim]
        return (p @ v.transpose(1, 2)).transpose(1, 2).reshape(b, n, -1)

    def latent(p, mx, h):
        rank, r = mx["kv_rank"], mx.get("rot_dim", 0)
        low = h @ w(p + "dkv").T
        c = _rms(low[..., :rank], eps) * w(p + "dkv.norm")
        k, v = split(c @ w(p + "uk").T, heads), split(c @ w(p + "uv").T, heads)
        q = split((_rms(h @ w(p + "dq").T, eps) * w(p + "dq.norm")) @ w(p + "uq").T if "q_rank" in mx else h @ w(p + "q").T, heads)
        s = q[..., :dim].transpose(1, 2) @ k.permute(0, 2, 3, 1)
        if r:
            rot = mx["rot"]
            kr = _turn(low[..., None, rank:], pos, rot["dims"], rot["base"], False)
            s = s + _turn(q[..., dim:], pos, rot["dims"], rot["base"], False).transpose(1, 2) @ kr.permute(0, 2, 3, 1)
        a = attend(_softmax_with((s * mx["scale"]).masked_fill(~causal, -math.inf), w(p + "sink").view(1, -1, 1, 1)), v)
        return (a * torch.sigmoid(h @ w(p + "g").T) if r else a) @ w(p + "o").T

    def lightning(p, mx, h):
        q, k, v = (split(torch.nn.functional.silu(h @ w(p + c).T), heads) for c in "qkv")
        decay = torch.tensor(mx["decay"], device="cuda", dtype=torch.float64).view(-1, 1, 1) ** (pos[:, None] - pos[None, :]).clamp(min=0)
        a = attend((q.transpose(1, 2) @ k.permute(0, 2, 3, 1) * decay).masked_fill(~causal, 0.0), v)
        return (_rms(a, eps) * w(p + "norm") * torch.sigmoid(h @ w(p + "g").T)) @ w(p + "o").T

    def routed(p, mlp, h):
        r = mlp["router"]
        s = torch.softmax(h @ w(p + "router").T, -1)
        chosen = torch.zeros_like(s).scatter_(-1, (s + w(p + "correction")).topk(r["top"], -1).indices, 1.0) * s
        out = chosen[..., r["experts"]:].sum(-1, keepdim=True) * h
        for e in range(r["experts"]):
            out = out + chosen[..., e:e + 1] * (torch.relu(h @ w(p + "e%d.up" % e).T) ** 2 @ w(p + "e%d.down" % e).T)
        return out

    def differential(p, mx, h):
        g, d = mx["kv_heads"], mx["dim"]
        q, k, v = (_conv(w(p + c + ".conv"), h @ w(p + c).T) for c in "qkv")
        rot = mx["rot"]
        q, k = (_turn(split(x, 2 * y), pos, rot["dims"], rot["base"], True).view(b, n, y, 2, d) for x, y in ((q, heads), (k, g)))
        k, v = k.repeat_interleave(heads // g, 2), split(v, g).repeat_interleave(heads // g, 2)
        sees = causal & ((pos[:, None] - pos[None, :] < mx["mask"]["size"]) | (pos[None, :] < mx["mask"]["keep_first"]))
        lam = torch.exp(w(p + "lq1") @ w(p + "lk1")) - torch.exp(w(p + "lq2") @ w(p + "lk2")) + mx["diff"]
        a = [attend(torch.softmax((q[..., m, :].transpose(1, 2) @ k[..., m, :].permute(0, 2, 3, 1) * mx["scale"]).masked_fill(~sees, -math.inf), -1), v) for m in (0, 1)]
        return (_rms(split(a[0] - lam * a[1], heads), eps) * (1.0 - mx["diff"])).reshape(b, n, -1) @ w(p + "o").T

    def delta(p, mx, h):
        g = mx["kv_heads"]
        q, k, v = (torch.nn.functional.silu(_conv(w(p + c + ".conv"), h @ w(p + c).T)) for c in "qkv")
        unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        q, k = (unit(split(x, g)).repeat_interleave(heads // g, 2) for x in (q, k))
        v, beta = split(v, heads), torch.sigmoid(h @ w(p + "b").T)
        keep = torch.exp(-torch.exp(w(p + "A_log"))[:, None] * torch.nn.functional.softplus(split(h @ w(p + "a1").T @ w(p + "a2").T + w(p + "dt_bias"), heads)))
        S, out = torch.zeros(b, heads, dim, vdim, device="cuda", dtype=torch.float64), []
        for i in range(n):
            S = S * keep[:, i, :, :, None]
            u = beta[:, i, :, None] * (v[:, i] - (k[:, i, :, None] @ S)[..., 0, :])
            S = S + k[:, i, :, :, None] * u[:, :, None, :]
            out.append((q[:, i, :, None] @ S)[..., 0, :])
        gate = torch.sigmoid(h @ w(p + "g1").T @ w(p + "g2").T)
        return ((_rms(torch.stack(out, 1) * dim ** -0.5, eps) * w(p + "norm")).reshape(b, n, -1) * gate) @ w(p + "o").T

    def chunked(p, mx, h):
        g, rot = mx["kv_heads"], mx["rot"]
        q, k = (_rms(_turn(split(h @ w(p + c).T, y), pos, rot["dims"], rot["base"], True), eps) for c, y in (("q", heads), ("k", g)))
        k, v = k.repeat_interleave(heads // g, 2), split(h @ w(p + "v").T, g).repeat_interleave(heads // g, 2)
        sees = causal & (pos[:, None] // mx["mask"]["size"] == pos[None, :] // mx["mask"]["size"])
        s = mx["softcap"] * torch.tanh(q.transpose(1, 2) @ k.permute(0, 2, 3, 1) * mx["scale"] / mx["softcap"])
        e = torch.exp(s).masked_fill(~sees, 0.0)
        return attend(e / (1.0 + e.sum(-1, keepdim=True)), v) @ w(p + "o").T

    def time_mix(p, mx, h):
        hs, d = mx["heads"], mx["dim"]
        before = torch.nn.functional.pad(h, (0, 0, 1, 0))[:, :n]
        m = {c: h + (before - h) * w(p + "mu." + c) for c in "rkvgw"}
        r, k, v = (split(m[c] @ w(p + c).T, hs) for c in "rkv")
        keep = torch.exp(-torch.exp(split(torch.tanh(m["w"] @ w(p + "w1").T) @ w(p + "w2").T + w(p + "w0"), hs)))
        S, out = torch.zeros(b, hs, d, d, device="cuda", dtype=torch.float64), []
        for i in range(n):
            kv = k[:, i, :, :, None] * v[:, i, :, None, :]
            out.append((r[:, i, :, None] @ (S + w(p + "u")[:, :, None] * kv))[..., 0, :])
            S = S * keep[:, i, :, :, None] + kv
        return (_rms(torch.stack(out, 1), eps).reshape(b, n, -1) * w(p + "norm") * torch.nn.functional.silu(m["g"] @ w(p + "g").T)) @ w(p + "o").T

    def pair_rows():
        pr = cfg["embedding"]["bigram"]
        rows = torch.full_like(ids, pr["buckets"])
        rows[:, 1:] = (ids[:, :-1] * pr["mul_prev"] + ids[:, 1:] * pr["mul_cur"]) % pr["buckets"]
        return tensors["bigram"][rows].double()

    design, x = cfg["architecture"], tensors["embed"][ids].double()
    if design != "Fasovik":
        x = x + pair_rows()
    for i, layer in enumerate(cfg["layers"]):
        p, q, mx = "l%d." % i, "l%d.mix." % i, layer["mixer"]
        if design == "Fasovik":
            x = x + cfg["residual_mult"] * _rms((lightning if layer["type"] == "lightning" else latent)(q, mx, x), eps) * (1.0 + w(p + "norm1"))
            x = x + cfg["residual_mult"] * _rms(routed(p + "mlp.", layer["mlp"], x), eps) * (1.0 + w(p + "norm2"))
        elif design == "Rafusun":
            if layer["type"] == "channel_delta":
                y = delta(q, mx, x)
            else:
                y = 0.5 * (_rms(chunked(q + "left.", mx["left"], x), eps) * w(q + "left.out") + _rms(time_mix(q + "right.", mx["right"], x), eps) * w(q + "right.out"))
            x = _rms(cfg["postln_alpha"] * x + w(p + "ls1") * y, eps) * w(p + "norm1")
            if layer["mlp"]:
                y = (torch.nn.functional.gelu(x @ w(p + "mlp.gate").T, approximate="tanh") * (x @ w(p + "mlp.up").T)) @ w(p + "mlp.down").T
                x = _rms(cfg["postln_alpha"] * x + w(p + "ls2") * y, eps) * w(p + "norm2")
        else:
            if i == cfg["loop"]["start"]:
                x = x + w("loop.step")[0]
            x = x + (differential if layer["type"] == "attention" else latent)(q, mx, _rms(x, eps) * w(p + "norm1"))
            h, limit = _rms(x, eps) * w(p + "norm2"), layer["mlp"]["limit"]
            u, v = (h @ w(p + "mlp.gate").T).clamp(max=limit), (h @ w(p + "mlp.up").T).clamp(-limit, limit)
            x = x + (u * torch.sigmoid(1.702 * u) * (v + 1.0)) @ w(p + "mlp.down").T
    x = _rms(x, eps) * (1.0 + w("final.norm") if design == "Fasovik" else w("final.norm"))
    head = w("head" if "head" in tensors else "embed").T

    def logits(rows):
        return (rows @ head).cpu().numpy()
    p0, at = case["past"], case["past"] + case["prompt"]
    out = [logits((x[:, p0:at] if case["score"] else x[:, at - 1:at]).reshape(-1, x.shape[-1]))] if case["prompt"] else []
    return out + [logits(x[:, at + k]) for k in range(case["steps"])]


def exact(case, seed):
    with torch.no_grad():
        return _exact_quant(case, seed) if case["kind"] == "quant" else _exact_folder(case, seed)
