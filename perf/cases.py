"""The work that users of this engine have it do, as cases that can be timed and compared.

A case is one pass through the engine's step function (`ModelRunner.step`) on a model with random
weights, or one call of its sampler. `batch` requests that hold about `context` tokens each bring
one token (decoding); `prompts` new requests bring `tokens` prompt tokens between them; a step may
mix both, as the scheduler's steps do. Model sizes are those of the benchmark: Qwen1.5-MoE-A2.7B
shapes and the "small" and "medium" sizes of the six other designs.
"""
from __future__ import annotations

import math
import random
import re
from typing import Dict, List, Optional

import numpy as np
import torch

import ninfer_amd
from ninfer_amd import Chunk, EngineOptions, ModelRunner, Sampler, SamplingParams, build_spec
from ninfer_amd.kernels import load_ops
from ninfer_amd.sampling import SampleRow
from ninfer_amd.sampling.sampler import History
from ninfer_amd.weights.source import RandomSource

D = torch.float64
ROOM = 1024          # tokens a decoding request generates before its place is taken by a new one
FILL = 2048          # tokens of a step that brings contexts into the cache
EXACT_FLOPS = 4.5e14   # more than this in 64 bits takes too long


# ---- models ------------------------------------------------------------------------------------

QWEN = {
    "architectures": ["Qwen2MoeForCausalLM"], "model_type": "qwen2_moe",
    "num_hidden_layers": 24, "hidden_size": 2048, "num_attention_heads": 16,
    "num_key_value_heads": 16, "head_dim": 128, "intermediate_size": 5632,
    "moe_intermediate_size": 1408, "shared_expert_intermediate_size": 5632,
    "num_experts": 60, "num_experts_per_tok": 4, "norm_topk_prob": False,
    "decoder_sparse_step": 1, "mlp_only_layers": [], "vocab_size": 151936,
    "rope_theta": 1000000.0, "use_sliding_window": False, "rms_norm_eps": 1e-6,
    "tie_word_embeddings": False, "hidden_act": "silu",
}
SMALL = dict(width=1024, ff=2816, heads=8, kv=2, experts=16, top=2, expert_ff=704)
MEDIUM = dict(width=2048, ff=5632, heads=16, kv=4, experts=32, top=4, expert_ff=1408)


def getodra(z: dict, medium: bool) -> dict:
    rot = 64 if medium else 32
    vdim = 128 if medium else 64
    latent = {"heads": z["heads"], "dim": 128 - rot, "rot_dim": rot, "vdim": vdim,
              "kv_rank": 512 if medium else 256, "scale": 128 ** -0.5,
              "rot": {"base": 10000.0, "dims": rot,
                      "scaling": {"factor": 8.0, "original": 1024, "fast": 16.0, "slow": 2.0}}}
    lightning = {"heads": z["heads"], "dim": 128, "vdim": vdim,
                 "decay": [1.0 - 2.0 ** -(3 + 5 * h / (z["heads"] - 1)) for h in range(z["heads"])]}
    layers = []
    for i in range(8):
        kind, mixer = ("lightning", lightning) if i % 4 == 0 else ("latent_attention", latent)
        layers.append({"type": kind, "mixer": mixer, "mlp": {"kind": "dense", "ff": z["ff"]}})
        if i % 4 == 2:
            layers[-1]["weights_of"] = i - 1
    return {"architecture": "Getodra", "vocab": 32000, "width": z["width"], "max_positions": 4096,
            "norm": {"eps": 1e-5}, "canon": {"taps": 4}, "layers": layers}


def sosepel(z: dict, medium: bool) -> dict:
    mixer = {"heads": z["heads"], "kv_heads": z["kv"], "dim": 64, "vdim": 128, "diff": 0.5,
             "scale": 64 ** -0.5, "softcap": 30.0, "q_temp": {"coef": 0.25, "every": 128}}
    moe = {"kind": "moe", "expert": {"ff": z["expert_ff"]}, "shared": {"ff": 2 * z["expert_ff"]},
           "router": {"experts": z["experts"], "top": z["top"], "groups": {"count": 4, "keep": 2}}}
    n = 6 if medium else 5
    layers = [{"type": "attention", "mixer": mixer,
               "mlp": moe if i else {"kind": "dense", "ff": z["ff"]}} for i in range(n)]
    return {"architecture": "Sosepel", "vocab": 32000, "width": z["width"], "norm": {"eps": 1e-6},
            "logit_softcap": 20.0, "embedding": {"scale": 50.0, "bigram": {
                "buckets": 65521, "mul_prev": 31, "mul_cur": 3}},
            "layers": layers, "loop": {"start": 1, "stop": n - 1, "times": 2}}


def fopinex(z: dict, medium: bool) -> dict:
    attention = {"heads": z["heads"], "kv_heads": z["kv"], "dim": 128, "vdim": 128,
                 "scale": 128 ** -0.5, "mask": {"size": 1024}}
    gla = {"heads": z["heads"], "dim": 64, "vdim": 128, "tau": 8.0, "rank": 64 if medium else 32}
    moe = {"kind": "moe", "expert": {"ff": z["expert_ff"], "limit": 7.0},
           "router": {"experts": z["experts"], "identity": 4 if medium else 2, "top": z["top"],
                      "groups": {"count": 4 if medium else 3, "keep": 2}}}
    layers = []
    for i in range(8):
        if i % 4 == 1:
            layers.append({"type": "gla", "mixer": gla, "mlp": moe})
        else:
            mixer = dict(attention, kv_from=i - 2) if i % 4 == 2 else attention
            layers.append({"type": "attention", "mixer": mixer, "mlp": moe})
    return {"architecture": "Fopinex", "vocab": 32000, "width": z["width"], "norm": {"eps": 1e-6},
            "residual_mult": 0.7, "layers": layers}


def tuzapel(z: dict, medium: bool) -> dict:
    rot = 64 if medium else 32
    attention = {"heads": z["heads"], "kv_heads": z["kv"], "dim": 128, "vdim": 128,
                 "scale": 128 ** -0.5, "conv": 4, "mask": {"size": 1024},
                 "rot": {"base": 500000.0, "dims": 64,
                         "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 2048}}}
    latent = {"heads": z["heads"], "dim": 128 - rot, "rot_dim": rot, "vdim": 128 if medium else 64,
              "kv_rank": 512 if medium else 256, "q_rank": 768 if medium else 384,
              "scale": 128 ** -0.5, "rot": {"base": 10000.0, "dims": rot}}
    moe = {"kind": "moe", "expert": {"ff": z["expert_ff"], "limit": 7.0},
           "router": {"experts": z["experts"], "top": z["top"]}}
    dense = {"kind": "dense", "ff": z["ff"], "limit": 7.0}
    layers = []
    for i in range(8):
        mlp = moe if i % 2 else dense
        if i % 4 == 0:
            layers.append({"type": "latent_attention", "mixer": latent, "mlp": mlp})
        else:
            mixer = dict(attention, kv_from=i - 1) if i % 4 == 2 else attention
            layers.append({"type": "attention", "mixer": mixer, "mlp": mlp})
    return {"architecture": "Tuzapel", "vocab": 32000, "width": z["width"], "norm": {"eps": 1e-6},
            "logit_softcap": 30.0, "layers": layers}


def rudazen(z: dict, medium: bool) -> dict:
    attention = {"heads": z["heads"], "kv_heads": z["kv"], "dim": 128, "vdim": 128,
                 "scale": 128 ** -0.5, "rot": {"base": 500000.0, "dims": 128}}
    pooled = dict(attention, mask={"size": 1024, "pool": 16})
    left = dict(attention, mask={"size": 1024}, rot={
        "base": 10000.0, "dims": 64,
        "scaling": {"factor": 8.0, "original": 2048, "fast": 32.0, "slow": 1.0}})
    right = {"heads": z["heads"], "dim": 64, "vdim": 128}
    mlp = {"kind": "dense", "ff": z["ff"]}
    layers = [{"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": mlp}
              if i % 4 == 2 else {"type": "attention", "mixer": pooled, "mlp": mlp}
              for i in range(8)]
    return {"architecture": "Rudazen", "vocab": 32000, "width": z["width"], "norm": {"eps": 1e-6},
            "postln_alpha": 2.0, "embedding": {"scale": z["width"] ** 0.5}, "layers": layers}


def nosedra(z: dict, medium: bool) -> dict:
    mlp = {"kind": "dense", "ff": z["ff"]}
    left = {"heads": z["heads"], "kv_heads": z["kv"], "dim": 128, "vdim": 128,
            "scale": 128 ** -0.5,
            "rot": {"base": 500000.0, "dims": 64, "scaling": {"factor": 4.0}}}
    right = {"heads": z["heads"] // 2, "dim": 128, "vdim": 256, "gate_cap": 15.0}
    both = {"type": "parallel", "mlp": mlp,
            "mixer": {"left": left, "left_scale": 0.7, "right_scale": 0.7, "right": right}}
    ssm = {"type": "mamba2", "mlp": mlp,
           "mixer": {"heads": 64 if medium else 32, "vdim": 64, "state": 128,
                     "groups": 8 if medium else 4, "conv": 4, "norm_groups": 1}}
    return {"architecture": "Nosedra", "vocab": 32000, "width": z["width"], "norm": {"eps": 1e-6},
            "logit_softcap": 30.0, "token_side": {"dim": 256 if medium else 128},
            "layers": [ssm if i % 4 == 1 else both for i in range(8)]}


DESIGNS = {f.__name__: f for f in (getodra, sosepel, fopinex, tuzapel, rudazen, nosedra)}


def config(model: str) -> dict:
    if model == "qwen2-moe":
        return QWEN
    name, size = model.split("-")
    return DESIGNS[name](MEDIUM if size == "medium" else SMALL, size == "medium")


# ---- the cases ---------------------------------------------------------------------------------

def _step(name: str, model: str, batch: int = 0, context: int = 0, prompts: int = 0,
          tokens: int = 0, dtype: str = "bfloat16", graph: bool = False) -> dict:
    return {"name": name, "kind": "step", "model": model, "dtype": dtype, "batch": batch,
            "context": context, "prompts": prompts, "tokens": tokens, "graph": graph}


def listed() -> List[dict]:
    return [
        # one user's chat: a token at a time, where launches and latency are what is paid for
        _step("chat decode", "qwen2-moe", batch=1, context=900, graph=True),
        # the benchmark's headline: a few users with long contexts
        _step("decode 8 long", "qwen2-moe", batch=8, context=7900, graph=True),
        # a full server: many users, ordinary contexts
        _step("decode 64", "qwen2-moe", batch=64, context=1900, graph=True),
        # the benchmark's prompt
        _step("prompt 2048", "qwen2-moe", prompts=1, tokens=2048),
        # a step of the scheduler at its default budget of 512 tokens: users that decode beside
        # the odd rest of somebody's prompt
        _step("mixed 512", "qwen2-moe", batch=7, context=2500, prompts=1, tokens=505),
        # the 32-bit path, as --verify runs a prompt again
        _step("verify 32-bit", "qwen2-moe", prompts=1, tokens=173, dtype="float32"),
        # the sampler behind a full server's step, with the default options
        {"name": "sample 64", "kind": "sample", "rows": 64, "vocab": 151936, "temperature": 0.7,
         "top_k": 50, "top_p": 0.95, "penalty": 1.05, "history": 1500},
        # the other designs, each in another of these uses
        _step("getodra prompt", "getodra-medium", prompts=1, tokens=2048),
        _step("sosepel prompts", "sosepel-medium", prompts=3, tokens=1531),
        _step("fopinex decode 8", "fopinex-medium", batch=8, context=2800, graph=True),
        _step("tuzapel decode 64", "tuzapel-medium", batch=64, context=2600, graph=True),
        _step("nosedra mixed", "nosedra-medium", batch=16, context=1500, prompts=2, tokens=1100),
    ]


def _log_int(rng: random.Random, low: int, high: int) -> int:
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng: random.Random) -> dict:
    """The same uses over their ranges: one to 64 decoding requests with contexts of 64 to 7,900
    tokens, prompts of 16 to 2,048 tokens in up to four requests, both in one step; every
    design in both sizes; 32-bit for small steps; the sampler with its options."""
    what = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "32-bit", "sample"])
    if what == "sample":
        sampled = rng.random() < 0.8
        return {"kind": "sample", "rows": _log_int(rng, 1, 64),
                "vocab": rng.choice([32000, 151936]),
                "temperature": round(rng.uniform(0.3, 1.2), 2) if sampled else 0.0,
                "top_k": rng.choice([0, 20, 50, 200]), "top_p": rng.choice([0.8, 0.95, 1.0]),
                "penalty": rng.choice([1.0, 1.05]), "history": _log_int(rng, 16, 2000)}
    model = "qwen2-moe" if rng.random() < 0.4 else \
        f"{rng.choice(sorted(DESIGNS))}-{rng.choice(['small', 'medium'])}"
    case = _step("", model)
    del case["name"]
    if what == "32-bit":
        # no longer than the listed one: the widest model costs most there
        case.update(dtype="float32", prompts=1, tokens=_log_int(rng, 16, 150))
        return case
    if what != "prompt":
        case["batch"] = _log_int(rng, 1, 64 if what == "decode" else 24)
        longest = 7900 if model == "qwen2-moe" else 2900
        # as many cached tokens as the listed cases have at most
        case["context"] = _log_int(rng, 64, min(longest, 120000 // case["batch"]))
        case["graph"] = what == "decode" and rng.random() < 0.7
    if what != "decode":
        case["tokens"] = _log_int(rng, 16, 2048 if what == "prompt" else 1100)
        case["prompts"] = rng.randint(1, min(4, case["tokens"] // 8))
    return case


def _contexts(case: dict) -> List[int]:
    """Tokens each decoding request holds: up to a quarter fewer than the case's context."""
    spread = case["context"] // 4 + 1
    return [case["context"] - (37 * i) % spread for i in range(case["batch"])]


def _prompts(case: dict) -> List[int]:
    """The lengths of a case's prompts: uneven parts of its tokens."""
    n, left, out = case["prompts"], case["tokens"], []
    for i in range(n):
        part = left if i == n - 1 else max(1, left * 3 // (5 * (n - i)) + 1)
        out.append(part)
        left -= part
    return out


def _max_context(case: dict) -> int:
    return max([c + ROOM for c in _contexts(case)] + _prompts(case))


# ---- one pass ----------------------------------------------------------------------------------

class _Weights(RandomSource):
    """Random weights whose model rounds as a trained one does: a residual stream that no single
    layer dominates (embeddings of about unit size, matrices of 0.014) and routers that prefer
    some experts clearly (softmax routers eight times as large), so that where bfloat16 rounding
    turns the choice between two nearly equal experts, little hangs on it."""

    def __init__(self, spec, seed: int, dtype: str):
        self.sosepel = "loop.in" in spec.tensor_specs()
        self.tied = not {"head", "lm_head.weight"} & set(spec.tensor_specs())
        super().__init__(spec.tensor_specs(), seed, getattr(torch, dtype), std=0.014, device="cuda:0")

    def read(self, name: str) -> torch.Tensor:
        t = super().read(name)
        if name in ("embed", "pos", "model.embed_tokens.weight") and not self.tied:
            t *= 50
        elif name.endswith((".router", ".mlp.gate.weight")) and not self.sosepel:
            t *= 8
        return t


class _Serving:
    """An engine with its decoding requests, and the prompts that new requests bring."""

    def __init__(self, case: dict, seed: int):
        self.case = case
        slots = case["batch"] + case["prompts"]
        options = EngineOptions(dtype=case["dtype"], max_context=_max_context(case),
                                prefill_chunk=FILL, num_sequences=slots, page_size=16,
                                use_graph=case["graph"])
        spec = build_spec(config(case["model"]))[1]
        self.runner = ModelRunner(spec, _Weights(spec, seed, case["dtype"]), options)
        rng = np.random.RandomState(seed % (1 << 32))
        vocab = self.runner.vocab_size
        self.contexts = [rng.randint(0, vocab, n).tolist() for n in _contexts(case)]
        self.prompts = [rng.randint(0, vocab, n).tolist() for n in _prompts(case)]
        self.next = rng.randint(0, vocab, (ROOM, max(1, case["batch"]))).tolist()
        self.slots: List[int] = []

    def fill(self) -> None:
        """Decoding requests (again) in place of those that are done, contexts in the cache."""
        for s in self.slots:
            self.runner.close(s)
        self.slots = [self.runner.open() for _ in self.contexts]
        self.at = 0
        step: List[Chunk] = []
        left = FILL
        for slot, tokens in zip(self.slots, self.contexts):
            i = 0
            while i < len(tokens):
                n = min(left, len(tokens) - i)
                step.append(Chunk(slot, tokens[i:i + n], []))
                i, left = i + n, left - n
                if left == 0:
                    self.runner.step(step)
                    step, left = [], FILL
        if step:
            self.runner.step(step)

    def __del__(self):
        if hasattr(self, "runner"):
            self.runner.release()


class _Sampling:
    def __init__(self, case: dict, seed: int):
        device = torch.device("cuda:0")
        gen = torch.Generator(device).manual_seed(seed)
        # logits as peaked as a trained model's: a few tokens of a row carry most of its mass
        self.logits = 3.0 * torch.randn(case["rows"], case["vocab"], generator=gen, device=device)
        self.sampler = Sampler(load_ops(), device)
        rng = np.random.RandomState(seed % (1 << 32))
        params = SamplingParams(temperature=case["temperature"], top_k=case["top_k"],
                                top_p=case["top_p"], repetition_penalty=case["penalty"], seed=1)
        self.rows = [SampleRow(params, History(rng.randint(0, case["vocab"], case["history"])),
                               key=i, draw=0, seed=seed + 1) for i in range(case["rows"])]


def prepare(case: dict, seed: int):
    if case["kind"] == "sample":
        return _Sampling(case, seed)
    state = _Serving(case, seed)
    state.fill()
    return state


def run(state):
    """Tokens of the sampler, or the step's logits at the last token of every request."""
    if isinstance(state, _Sampling):
        return np.asarray(state.sampler.sample(state.logits, state.rows), dtype=np.int64)
    runner = state.runner
    if state.at == ROOM:
        state.fill()
    chunks = [Chunk(s, [t], [0]) for s, t in zip(state.slots, state.next[state.at])]
    state.at += 1
    new = [runner.open() for _ in state.prompts]
    chunks += [Chunk(s, p, [len(p) - 1]) for s, p in zip(new, state.prompts)]
    logits = runner.step(chunks)
    for s in new:
        runner.close(s)
    return logits


# ---- what a pass cannot do without ---------------------------------------------------------------

def _layer_runs(cfg: dict) -> List[tuple]:
    """(layer, layer whose tensors it runs) of every run of a layer, in order."""
    if "layers" not in cfg:
        return [(i, i) for i in range(cfg["num_hidden_layers"])]
    loop = cfg.get("loop")
    n = len(cfg["layers"])
    order = list(range(n)) if not loop else list(range(loop["start"])) + \
        list(range(loop["start"], loop["stop"])) * loop["times"] + list(range(loop["stop"], n))
    return [(i, cfg["layers"][i].get("weights_of", i)) for i in order]


def _attention(cfg: dict) -> List[tuple]:
    """(numbers cached per token, operations per row and key, span of keys or None) of every
    layer run with attention, in the form that needs least."""
    if "layers" not in cfg:
        heads, kv, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
        return [(2 * kv * d, 4 * heads * d, None)] * cfg["num_hidden_layers"]
    out = []
    for i, _ in _layer_runs(cfg):
        layer = cfg["layers"][i]
        m = layer["mixer"].get("left", layer["mixer"])
        if layer["type"] == "latent_attention":
            out.append((m["kv_rank"] + m["rot_dim"],
                        2 * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), None))
        elif layer["type"] in ("attention", "parallel"):
            maps = 2 if "diff" in m else 1
            own = 0 if "kv_from" in m else m["kv_heads"] * (maps * m["dim"] + m["vdim"])
            out.append((own, 2 * m["heads"] * maps * (m["dim"] + m["vdim"]),
                        (m.get("mask") or {}).get("size")))
    return out


def _state_numbers(cfg: dict) -> int:
    """Numbers of per-request state of the recurrences."""
    total = 0
    for i, _ in _layer_runs(cfg) if "layers" in cfg else []:
        layer = cfg["layers"][i]
        m = layer["mixer"].get("right", layer["mixer"])
        if layer["type"] in ("lightning", "gla", "parallel"):
            total += m["heads"] * m["dim"] * m["vdim"]
        elif layer["type"] == "mamba2":
            total += m["heads"] * m["state"] * m["vdim"]
    return total


EXPERT = re.compile(r"\.(experts\.|e)\d+\.")


def work(case: dict) -> Dict[str, float]:
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4.0 * n, "flops": 2.0 * n}
    cfg = config(case["model"])
    size = 2 if case["dtype"] == "bfloat16" else 4
    spec = build_spec(cfg)[1]
    contexts, prompts = _contexts(case), _prompts(case)
    rows, wanted = len(contexts) + sum(prompts), len(contexts) + len(prompts)
    if "layers" not in cfg:
        experts, top, head, tables = cfg["num_experts"], cfg["num_experts_per_tok"], \
            "lm_head.weight", ("model.embed_tokens.weight",)
        place = r"model\.layers\.(\d+)\."
    else:
        router = next((l["mlp"]["router"] for l in cfg["layers"] if "router" in l["mlp"]), {})
        experts, top = router.get("experts", 1), router.get("top", 1)
        head = "embed" if cfg["architecture"] in ("Sosepel", "Tuzapel") else "head"
        tables = tuple({"embed", "pos", "bigram", "side.embed"} - {head})
        place = r"l(\d+)\."
    runs = [j for _, j in _layer_runs(cfg)]
    used = experts * (1 - (1 - top / experts) ** rows)     # experts met by rows that choose evenly
    nbytes = flops = 0.0
    for name, t in spec.tensor_specs().items():
        if name in tables or len(t.shape) < 2:
            continue
        n = float(np.prod(t.shape))
        if name == head:
            nbytes, flops = nbytes + n * size, flops + 2 * n * wanted
            continue
        at = re.match(place, name)
        times = runs.count(int(at.group(1))) if at else 1
        share, met = (top / experts, used / experts) if EXPERT.search(name) else (1.0, 1.0)
        nbytes += n * size * met
        flops += 2 * n * rows * share * times
    for numbers, each, span in _attention(cfg):
        for c in contexts:
            seen = min(c + 1, span or c + 1)
            nbytes, flops = nbytes + seen * numbers * size, flops + seen * each
        for p in prompts:
            keys = sum(min(i + 1, span or p) for i in range(p))
            nbytes, flops = nbytes + p * numbers * size, flops + keys * each
    state = _state_numbers(cfg)
    nbytes += 4 * state * (2 * len(contexts) + len(prompts)) + 4 * wanted * spec.vocab_size
    flops += 4 * state * rows
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict):
    """In 32-bit the listed case is 3e-6 off its 64-bit value. In bfloat16 the designs are 0.003 to
    0.014 off, and 0.02 to 0.03 where one row of a few has another expert chosen."""
    if case["kind"] == "sample":
        return "exact"
    return {"rel": 1.2e-5} if case["dtype"] == "float32" else {"rel": 0.03}


# ---- the same in 64 bits -------------------------------------------------------------------------

class _Plain:
    """Whole sequences in plain 64-bit torch, no cache: `x` is [requests, tokens, width], requests
    shorter than the longest end in padding that no earlier token sees."""

    def __init__(self, cfg: dict, tensor, tokens: torch.Tensor):
        self.cfg, self.tensor, self.tokens = cfg, tensor, tokens
        self.B, self.n = tokens.shape
        self.dev = tokens.device
        self.pos = torch.arange(self.n, device=self.dev, dtype=D)
        self.eps = cfg["rms_norm_eps"] if "rms_norm_eps" in cfg else cfg["norm"]["eps"]

    def w(self, name: str) -> torch.Tensor:
        return self.tensor(name).to(D)

    def lin(self, name: str, x: torch.Tensor, bias: Optional[str] = None) -> torch.Tensor:
        y = x @ self.w(name).T
        return y + self.w(bias) if bias else y

    def rms(self, x: torch.Tensor, gain: Optional[str] = None) -> torch.Tensor:
        y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.eps)
        return y * self.w(gain) if gain else y

    def layer_norm(self, x: torch.Tensor, gain: str) -> torch.Tensor:
        return self.rms(x - x.mean(-1, keepdim=True), gain)

    def heads(self, x: torch.Tensor, heads: int) -> torch.Tensor:
        return x.reshape(self.B, self.n, heads, -1)

    def turn(self, x: torch.Tensor, freq: torch.Tensor, neighbours: bool = False,
             factor: float = 1.0) -> torch.Tensor:
        """x [B, n, heads, d]: its first numbers turn by position x frequency, in pairs of
        neighbours or of the two halves; the rest pass."""
        half = freq.numel()
        a = (self.pos[:, None] * freq.to(self.dev))[None, :, None, :]
        c, s = torch.cos(a) * factor, torch.sin(a) * factor
        first, second = (slice(0, 2 * half, 2), slice(1, 2 * half, 2)) if neighbours else \
            (slice(0, half), slice(half, 2 * half))
        u, v = x[..., first], x[..., second]
        y = x.clone()
        y[..., first], y[..., second] = u * c - v * s, v * c + u * s
        return y

    def conv(self, x: torch.Tensor, taps: torch.Tensor) -> torch.Tensor:
        y = torch.zeros_like(x)
        for j in range(taps.shape[1]):
            back = taps.shape[1] - 1 - j
            y[:, back:] += taps[:, j] * x[:, :self.n - back]
        return y

    def attend(self, q, k, v, scale: float, span: Optional[int] = None, weigh=None, more=None):
        """q [B, n, H, d] over k, v [B, n, G, .]: a row sees itself and the span - 1 tokens before
        it. `weigh` turns scores [H, rows, keys] and what is seen into weights (softmax if not
        given); `more`: (keys, values, last token of each) of blocks seen before the span."""
        H, G = q.shape[2], k.shape[2]
        at = self.pos
        out = torch.empty(*q.shape[:3], v.shape[-1], device=self.dev, dtype=D)
        weigh = weigh or (lambda s, seen: torch.softmax(s.masked_fill(~seen, -math.inf), -1))
        for b in range(self.B):
            for i in range(0, self.n, 512):
                j = min(self.n, i + 512)
                kb, vb = k[b, :j], v[b, :j]
                back = at[i:j, None] - at[None, :j]
                seen = (back >= 0) & (back < (span or self.n))
                if more is not None:
                    kb, vb = torch.cat([more[0][b], kb]), torch.cat([more[1][b], vb])
                    seen = torch.cat([more[2][None, :] <= at[i:j, None] - span, seen], 1)
                s = torch.einsum("rgpd,kgd->gprk", q[b, i:j].reshape(j - i, G, H // G, -1), kb)
                p = weigh(s.reshape(H, j - i, -1) * scale, seen[None])
                o = torch.einsum("gprk,kgd->rgpd", p.reshape(G, H // G, j - i, -1), vb)
                out[b, i:j] = o.reshape(j - i, H, -1)
        return out

    def scan(self, keep, k, v, q):
        """S = keep S + k v^T, o = S^T q, token by token; keep [B, n, H, 1 or d]."""
        S = torch.zeros(self.B, *k.shape[2:], v.shape[-1], device=self.dev, dtype=D)
        out = torch.empty_like(v)
        for t in range(self.n):
            S = keep[:, t, :, :, None] * S + k[:, t, :, :, None] * v[:, t, :, None, :]
            out[:, t] = (q[:, t, :, None, :] @ S)[..., 0, :]
        return out

    def experts(self, h, ids, weights, expert, real: int):
        flat = h.reshape(-1, h.shape[-1])
        y = torch.zeros_like(flat)
        for e in range(int(ids.max()) + 1):
            rows, choice = (ids == e).nonzero(as_tuple=True)
            if rows.numel():
                x = flat[rows]
                y[rows] += weights[rows, choice, None] * (expert(e, x) if e < real else x)
        return y.reshape(h.shape)

    def logits(self, wanted) -> torch.Tensor:
        """[wanted rows, vocab]; wanted: (request, token) of each."""
        x = getattr(self, self.cfg.get("architecture", "Qwen2Moe").lower())()
        b, t = torch.tensor(wanted, device=self.dev).T
        return self.head(x[b, t])

    # Qwen2-MoE
    def qwen2moe(self):
        c = self.cfg
        H, G, d = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        freq = c["rope_theta"] ** (-2.0 * torch.arange(d // 2, dtype=D) / d)
        x = self.w("model.embed_tokens.weight")[self.tokens]
        for l in range(c["num_hidden_layers"]):
            p = f"model.layers.{l}."
            h = self.rms(x, p + "input_layernorm.weight")
            q, k, v = (self.heads(self.lin(f"{p}self_attn.{i}_proj.weight", h,
                                           f"{p}self_attn.{i}_proj.bias"), m)
                       for i, m in (("q", H), ("k", G), ("v", G)))
            o = self.attend(self.turn(q, freq), self.turn(k, freq), v, d ** -0.5)
            x = x + self.lin(p + "self_attn.o_proj.weight", o.flatten(2))
            h = self.rms(x, p + "post_attention_layernorm.weight")

            def gated(prefix, h):
                return self.lin(prefix + "down_proj.weight",
                                torch.nn.functional.silu(self.lin(prefix + "gate_proj.weight", h))
                                * self.lin(prefix + "up_proj.weight", h))

            p += "mlp."
            prob = torch.softmax(self.lin(p + "gate.weight", h).flatten(0, 1), -1)
            wts, ids = prob.topk(c["num_experts_per_tok"], -1)
            x = x + self.experts(h, ids, wts, lambda e, y: gated(f"{p}experts.{e}.", y),
                                 c["num_experts"])
            x = x + torch.sigmoid(self.lin(p + "shared_expert_gate.weight", h)) \
                * gated(p + "shared_expert.", h)
        return x

    def head(self, x):
        c = self.cfg
        if "layers" not in c:
            return self.lin("lm_head.weight", self.rms(x, "model.norm.weight"))
        kind = c["architecture"]
        if kind == "Nosedra":
            x = self.rms(x) * (1.0 + self.w("final.norm"))
        else:
            x = (self.layer_norm if kind == "Tuzapel" else self.rms)(x, "final.norm")
        z = self.lin("embed" if kind in ("Sosepel", "Tuzapel") else "head", x)
        cap = c.get("logit_softcap")
        return cap * torch.tanh(z / cap) if cap else z

    def latent(self, p, m, h, q, neighbours, freq, factor=1.0):
        H, d, R = m["heads"], m["dim"], m["kv_rank"]
        q = self.heads(q, H)
        down = self.lin(p + "dkv", h)
        c = self.rms(down[..., :R], p + "dkv.norm")
        turned = self.turn(self.heads(down[..., R:], 1), freq, neighbours, factor)
        q = torch.cat([q[..., :d], self.turn(q[..., d:], freq, neighbours, factor)], -1)
        k = torch.cat([self.heads(self.lin(p + "uk", c), H), turned.expand(-1, -1, H, -1)], -1)
        return self.attend(q, k, self.heads(self.lin(p + "uv", c), H), m["scale"])

    @staticmethod
    def frequencies(rot: dict) -> torch.Tensor:
        return rot["base"] ** (-2.0 * torch.arange(rot["dims"] // 2, dtype=D) / rot["dims"])

    def stretched(self, rot: dict):
        """Frequencies slowed down in parts, and the factor on cosine and sine."""
        f, n, sc = self.frequencies(rot), rot["dims"], rot.get("scaling")
        if not sc:
            return f, 1.0
        lo, hi = (n * math.log(sc["original"] / (2 * math.pi * sc[k])) / (2 * math.log(rot["base"]))
                  for k in ("fast", "slow"))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), n - 1)
        ramp = ((torch.arange(n // 2, dtype=D) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0

    def getodra(self):
        x = self.w("embed")[self.tokens] + self.w("pos")[:self.n]
        for i, j in _layer_runs(self.cfg):
            p, m = f"l{j}.", self.cfg["layers"][i]["mixer"]
            h = x + self.conv(x, self.w(p + "canon1"))
            if self.cfg["layers"][i]["type"] == "lightning":
                q, k, v = (torch.nn.functional.silu(self.heads(self.lin(f"{p}mix.{a}", h), m["heads"]))
                           for a in "qkv")
                keep = torch.tensor(m["decay"], device=self.dev, dtype=D)[None, None, :, None]
                o = self.scan(keep.expand(self.B, self.n, -1, 1), k, v, q).flatten(2)
                y = self.rms(o, p + "mix.norm") * torch.sigmoid(self.lin(p + "mix.g", h))
            else:
                freq, factor = self.stretched(m["rot"])
                o = self.latent(p + "mix.", m, h, self.lin(p + "mix.q", h), False, freq, factor)
                y = (o * torch.sigmoid(self.lin(p + "mix.g", h))[..., None]).flatten(2)
            x = x + self.rms(self.lin(p + "mix.o", y)) * self.w(p + "norm1")
            h = x + self.conv(x, self.w(p + "canon2"))
            y = torch.nn.functional.gelu(self.lin(p + "mlp.gate", h), approximate="tanh") \
                * self.lin(p + "mlp.up", h)
            x = x + self.rms(self.lin(p + "mlp.down", y)) * self.w(p + "norm2")
        return x

    def sosepel(self):
        e = self.cfg["embedding"]
        x0 = self.w("embed")[self.tokens] * e["scale"]
        b = e["bigram"]
        pairs = (self.tokens[:, :-1] * b["mul_prev"] + self.tokens[:, 1:] * b["mul_cur"]) % b["buckets"]
        first = torch.full((self.B, 1), b["buckets"], device=self.dev)
        x0 = x0 + self.w("bigram")[torch.cat([first, pairs], 1)]
        x = x0
        for i, _ in _layer_runs(self.cfg):
            p, layer = f"l{i}.", self.cfg["layers"][i]
            m = layer["mixer"]
            if i == self.cfg["loop"]["start"]:
                x = self.lin("loop.in", torch.cat([x, x0], -1))
            h = self.rms(x, p + "norm1")
            q, k = (self.heads(self.lin(f"{p}mix.{a}", h), n).unflatten(-1, (2, -1))
                    for a, n in (("q", m["heads"]), ("k", m["kv_heads"])))
            v = self.heads(self.lin(p + "mix.v", h), m["kv_heads"])
            t = m["q_temp"]
            q = q * (1 + t["coef"] * torch.log(torch.floor((self.pos + 1) / t["every"]) + 1)
                     )[:, None, None, None]

            def weigh(s, seen):
                s = m["softcap"] * torch.tanh(s / m["softcap"])
                return torch.softmax(s.masked_fill(~seen, -math.inf), -1)

            a, c = (self.attend(q[..., j, :], k[..., j, :], v, m["scale"], weigh=weigh) for j in (0, 1))
            l = [self.w(p + "mix." + s) for s in ("lq1", "lk1", "lq2", "lk2")]
            lam = torch.exp(l[0] @ l[1]) - torch.exp(l[2] @ l[3]) + m["diff"]
            y = self.lin(p + "mix.o", (self.rms(a - lam * c) * (1 - m["diff"])).flatten(2))
            f = layer["mlp"]
            if f["kind"] == "dense":
                z = self.lin(p + "mlp.down", torch.relu(self.lin(p + "mlp.up", h)) ** 2)
            else:
                z = self.sosepel_sparse(p + "mlp.", f["router"], h)
            x = x + y * self.w(p + "ls1") + z * self.w(p + "ls2")
        return x

    def sosepel_sparse(self, p, r, h):
        def gated(prefix, y):
            return self.lin(prefix + "down", torch.nn.functional.silu(self.lin(prefix + "gate", y))
                            * self.lin(prefix + "up", y))

        s = torch.sigmoid(self.lin(p + "router", h).flatten(0, 1))
        groups = s.unflatten(-1, (r["groups"]["count"], -1))
        best = groups.topk(2, -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
        kept = torch.zeros(groups.shape[:2], device=self.dev, dtype=torch.bool).scatter_(1, best, True)
        wts, ids = torch.where(kept[..., None], groups, -1.0).flatten(1).topk(r["top"], -1)
        wts = wts / (wts.sum(-1, keepdim=True) + 1e-20)
        y = self.experts(h, ids, wts, lambda e, z: gated(f"{p}e{e}.", z), r["experts"])
        return y + torch.sigmoid(self.lin(p + "shared.sg", h)) * gated(p + "shared.", h)

    def clamped(self, prefix, limit, h):
        g = self.lin(prefix + "gate", h).clamp(max=limit)
        u = self.lin(prefix + "up", h).clamp(-limit, limit)
        return self.lin(prefix + "down", g * torch.sigmoid(1.702 * g) * (u + 1))

    def fopinex(self):
        x = self.w("embed")[self.tokens]
        kv = {}
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            H = m["heads"]
            h = self.rms(x, f"l{i}.norm1")
            if layer["type"] == "gla":
                q, k, v = (self.heads(self.lin(p + a, h), H) for a in "qkv")
                z = self.lin(p + "a2", self.lin(p + "a1", h), p + "a2.b")
                keep = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"])
                o = self.scan(self.heads(keep, H), k, v, q * m["dim"] ** -0.5)
                y = self.rms(o, p + "norm").flatten(2) * torch.nn.functional.silu(self.lin(p + "g", h))
            else:
                if "kv_from" not in m:
                    kv[i] = [self.heads(self.lin(p + a, h), m["kv_heads"]) for a in "kv"]
                k, v = kv[m.get("kv_from", i)]
                pb, talk, size = self.w(p + "pb"), self.w(p + "talk"), m["mask"]["size"]
                y = torch.empty(self.B, self.n, H, m["vdim"], device=self.dev, dtype=D)
                for a in range(0, self.n, size):     # a row sees its own chunk of positions
                    n = min(self.n, a + size) - a

                    def weigh(s, seen):
                        s = torch.sigmoid(s + pb[:, None, None]) * seen
                        return (talk @ s.flatten(1)).reshape(s.shape)

                    part = _Plain(self.cfg, self.tensor, self.tokens[:, a:a + n])
                    y[:, a:a + n] = part.attend(self.heads(self.lin(p + "q", h), H)[:, a:a + n],
                                                k[:, a:a + n], v[:, a:a + n], m["scale"], weigh=weigh)
                y = y.flatten(2)
            y = self.lin(p + "o", y) * torch.sigmoid(self.lin(f"l{i}.rg1", h, f"l{i}.rg1.b"))
            h = self.rms(x, f"l{i}.norm2")
            p, r = f"l{i}.mlp.", layer["mlp"]["router"]
            s = torch.softmax(self.lin(p + "router", h).flatten(0, 1), -1)
            choice = (s + self.w(p + "correction")).unflatten(-1, (r["groups"]["count"], -1))
            best = choice.max(-1).values.topk(r["groups"]["keep"], -1).indices
            kept = torch.zeros(choice.shape[:2], device=self.dev, dtype=torch.bool).scatter_(1, best, True)
            ids = torch.where(kept[..., None], choice, -math.inf).flatten(1).topk(r["top"], -1).indices
            limit = layer["mlp"]["expert"]["limit"]
            z = self.experts(h, ids, s.gather(-1, ids),
                             lambda e, t: self.clamped(f"{p}e{e}.", limit, t), r["experts"])
            y = y + z * torch.sigmoid(self.lin(f"l{i}.rg2", h, f"l{i}.rg2.b"))
            x = x + self.cfg["residual_mult"] * y
        return x

    def tuzapel(self):
        x = self.w("embed")[self.tokens]
        kv = {}
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            rot = m["rot"]
            freq = self.frequencies(rot)
            h = self.layer_norm(x, f"l{i}.norm1")
            if layer["type"] == "latent_attention":
                q = self.lin(p + "uq", self.rms(self.lin(p + "dq", h), p + "dq.norm"))
                o = self.latent(p, m, h, q, True, freq)
            else:
                sc = rot["scaling"]
                wave = 2 * math.pi / freq
                part = ((sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
                freq = (1 - part) * freq / sc["factor"] + part * freq

                def normed(a, heads):
                    y = self.heads(self.conv(self.lin(p + a, h), self.w(f"{p}{a}.conv")), heads)
                    return self.turn(self.rms(y, f"{p}{a}.norm"), freq)

                if "kv_from" not in m:
                    v = self.conv(self.lin(p + "v", h), self.w(p + "v.conv"))
                    kv[i] = normed("k", m["kv_heads"]), self.heads(v, m["kv_heads"])

                def weigh(s, seen):     # a sink: one more term exp(0) in the denominator
                    s = s.masked_fill(~seen, -math.inf)
                    sink = torch.zeros_like(s[..., :1])
                    return torch.softmax(torch.cat([s, sink], -1), -1)[..., :-1]

                o = self.attend(normed("q", m["heads"]), *kv[m.get("kv_from", i)], m["scale"],
                                m["mask"]["size"], weigh)
            x = x + self.layer_norm(self.lin(p + "o", o.flatten(2)), f"l{i}.norm1b")
            h = self.layer_norm(x, f"l{i}.norm2")
            p, f = f"l{i}.mlp.", layer["mlp"]
            if f["kind"] == "dense":
                y = self.clamped(p, f["limit"], h)
            else:
                z, ids = self.lin(p + "router", h, p + "router.b").flatten(0, 1).topk(f["router"]["top"], -1)
                y = self.experts(h, ids, torch.softmax(z, -1),
                                 lambda e, t: self.clamped(f"{p}e{e}.", f["expert"]["limit"], t),
                                 f["router"]["experts"])
            x = x + self.layer_norm(y, f"l{i}.norm2b")
        return x

    def rudazen(self):
        x = self.w("embed")[self.tokens] * self.cfg["embedding"]["scale"]
        alpha = self.cfg["postln_alpha"]
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]

            def normed(p, a, heads, rot, neighbours):
                freq, factor = self.stretched(rot)
                y = self.heads(self.rms(self.lin(p + a, x), f"{p}{a}.norm"), heads)
                return self.turn(y, freq, neighbours, factor)

            if layer["type"] == "attention":
                q = normed(p, "q", m["heads"], m["rot"], True)
                k = normed(p, "k", m["kv_heads"], m["rot"], True)
                v = self.heads(self.lin(p + "k", x), m["kv_heads"])
                pool = m["mask"]["pool"]
                whole = self.n // pool * pool
                means = [t[:, :whole].unflatten(1, (-1, pool)).mean(2) for t in (k, v)]
                last = torch.arange(self.n // pool, device=self.dev, dtype=D) * pool + pool - 1
                o = self.attend(q, k, v, m["scale"], m["mask"]["size"], more=(*means, last))
                y = self.lin(p + "o", o.flatten(2))
            else:
                a, r = m["left"], m["right"]
                q = normed(p + "left.", "q", a["heads"], a["rot"], False)
                k = normed(p + "left.", "k", a["kv_heads"], a["rot"], False)
                v = self.heads(self.lin(p + "left.v", x), a["kv_heads"])
                q = q * self.w(p + "left.temp")[:, None]
                o = self.attend(q, k, v, a["scale"], a["mask"]["size"]).flatten(2)
                left = self.lin(p + "left.o", o * torch.sigmoid(self.lin(p + "left.g", x)))
                lower = self.w(p + "right.lower")
                f = lower + (1 - lower) * torch.sigmoid(self.lin(p + "right.f", x, p + "right.f.b"))
                f = self.heads(f, r["heads"])
                q = self.heads(torch.nn.functional.silu(self.lin(p + "right.q", x)), r["heads"])
                o = self.scan(f, 1 - f, self.heads(self.lin(p + "right.v", x), r["heads"]), q)
                right = self.lin(p + "right.o", self.rms(o, p + "right.norm").flatten(2))
                y = 0.5 * (self.rms(left, p + "left.out") + self.rms(right, p + "right.out"))
            x = self.rms(alpha * x + y, f"l{i}.norm1")
            p = f"l{i}.mlp."
            y = self.lin(p + "down", torch.nn.functional.silu(self.lin(p + "gate", x))
                         * self.lin(p + "up", x))
            x = self.rms(alpha * x + y, f"l{i}.norm2")
        return x

    def nosedra(self):
        def gelu(z):
            return torch.nn.functional.gelu(z, approximate="tanh")

        side = self.cfg["token_side"]["dim"]
        x = self.w("embed")[self.tokens]
        for i, layer in enumerate(self.cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            h = self.rms(x) * (1 + self.w(f"l{i}.norm1"))
            x = x + (self.nosedra_ssm(p, m, h) if layer["type"] == "mamba2" else
                     m["left_scale"] * self.nosedra_attention(p + "left.", m["left"], h)
                     + m["right_scale"] * self.nosedra_memory(p + "right.", m["right"], h))
            h = self.rms(x) * (1 + self.w(f"l{i}.norm2"))
            p = f"l{i}.mlp."
            y = gelu(self.lin(p + "gate", h, p + "gate.b")) * self.lin(p + "up", h, p + "up.b")
            x = x + self.lin(p + "down", y, p + "down.b")
            p = f"l{i}.side."
            e = self.w("side.embed")[:, i * side:(i + 1) * side][self.tokens]
            x = x + self.rms(self.lin(p + "proj", gelu(self.lin(p + "gate", x)) * e), p + "norm")
        return x

    def nosedra_attention(self, p, m, h):
        freq = self.frequencies(m["rot"]) / m["rot"]["scaling"]["factor"]
        q, k = (self.rms(self.turn(self.heads(self.lin(p + a, h), n), freq))
                for a, n in (("q", m["heads"]), ("k", m["kv_heads"])))
        sink = self.w(p + "sink")[:, None, None]

        def weigh(s, seen):
            s = s.masked_fill(~seen, -math.inf)
            return torch.softmax(torch.cat([s, sink.expand(-1, s.shape[1], 1)], -1), -1)[..., :-1]

        o = self.attend(q, k, self.heads(self.lin(p + "v", h), m["kv_heads"]), m["scale"], weigh=weigh)
        return self.lin(p + "o", o.flatten(2) * torch.sigmoid(self.lin(p + "g", h)))

    def nosedra_memory(self, p, m, h):
        q, k, v = (self.heads(self.lin(p + a, h), m["heads"]) for a in "qkv")
        q = q * m["dim"] ** -0.5
        cap = m["gate_cap"]
        write = cap * torch.tanh(self.lin(p + "i", h, p + "i.b") / cap)
        keep = torch.nn.functional.logsigmoid(cap * torch.tanh(self.lin(p + "f", h, p + "f.b") / cap))
        top = torch.empty_like(write)
        now = torch.zeros(self.B, m["heads"], device=self.dev, dtype=D)
        for t in range(self.n):
            now = torch.maximum(keep[:, t] + now, write[:, t])
            top[:, t] = now
        before = torch.cat([torch.zeros_like(top[:, :1]), top[:, :-1]], 1)
        ones = torch.ones_like(v[..., :1])   # a further column of the state sums the keys alone
        o = self.scan(torch.exp(keep + before - top)[..., None],
                      torch.exp(write - top)[..., None] * k, torch.cat([v, ones], -1), q)
        den = torch.maximum(o[..., -1:].abs(), torch.exp(-top)[..., None]) + 1e-6
        o = self.rms(o[..., :-1] / den).flatten(2) * self.w(p + "norm")
        return self.lin(p + "o", o * torch.sigmoid(self.lin(p + "g", h)))

    def nosedra_ssm(self, p, m, h):
        H, G = m["heads"], m["groups"]
        inner, gn = H * m["vdim"], G * m["state"]
        z, xbc, dt = self.lin(p + "in", h).split([inner, inner + 2 * gn, H], -1)
        xbc = torch.nn.functional.silu(self.conv(xbc, self.w(p + "conv")) + self.w(p + "conv.b"))
        v, b, c = xbc.split([inner, gn, gn], -1)
        v = self.heads(v, H)
        b, c = (self.heads(t, G).repeat_interleave(H // G, 2) for t in (b, c))
        dt = torch.nn.functional.softplus(dt + self.w(p + "dt_bias"))
        keep = torch.exp(-torch.exp(self.w(p + "A_log")) * dt)
        y = self.scan(keep[..., None], dt[..., None] * b, v, c) + self.w(p + "D")[:, None] * v
        y = y.flatten(2) * torch.nn.functional.silu(z)
        y = self.rms(y.unflatten(-1, (m["norm_groups"], -1))).flatten(2) * self.w(p + "norm")
        return self.lin(p + "o", y)


def exact(case: dict, seed: int):
    """The logits of `run`'s first pass; its weights are read back by their names."""
    if case["kind"] == "sample":
        return None
    contexts = _contexts(case)
    whole = dict(case, batch=0, context=0, graph=False, prompts=1,
                 tokens=sum(contexts) + sum(_prompts(case)))
    if work(whole)["flops"] > EXACT_FLOPS:
        return None
    state = _Serving(case, seed)
    requests = [c + [t] for c, t in zip(state.contexts, state.next[0])] + state.prompts
    longest = max(len(r) for r in requests)
    tokens = torch.zeros(len(requests), longest, dtype=torch.long)
    for i, r in enumerate(requests):
        tokens[i, :len(r)] = torch.tensor(r)
    plain = _Plain(config(case["model"]), state.runner.tensor, tokens.to(state.runner.device))
    return plain.logits([(i, len(r) - 1) for i, r in enumerate(requests)])
