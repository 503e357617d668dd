"""The steps that this engine is used for, as cases that can be timed and compared.

A case is one call of ``ModelRunner.step``: ``singles`` requests that decode one token each behind
``context`` tokens, beside ``portions`` requests that bring ``portion`` tokens of a prompt each behind
``start`` tokens; ``rows`` positions of every portion want their logits (1: the last one, as generation
wants them; more: a prompt that is scored).  Lengths are ragged: request i is a little shorter than the
first, as the case's sizes alone say.  ``prepare`` builds the model with weights of the seed and brings
a program's requests to where the step starts; ``run`` is the step.

The models are the shapes that ``bench.py`` times: Llama at the 8B and the 1B shape and, at their m
size, four decoders that between them use every kind of layer that costs much: state-space and gated
recurrent layers (Dirulorn), matrix states with a decay a channel and with the delta rule beside routed
experts in groups (Vovalix), matrix memories with gates, windows and latent attention (Tazunex), routed
experts with a shared one behind attention that shares caches (Sopulorn).

Weights are drawn as trained models have them, so that rounding does not drown what is compared: a
sublayer adds a small part of the stream, gates and decays lie where such layers keep them.
"""

from __future__ import annotations

import math
import random
import zlib

import torch

DEVICE = "cuda:0"
PAGE = 16
MAX_LEN = 8192          # the context limit of the benchmark
FILL = 4096             # tokens a step while prepare() runs the earlier tokens
WARM = 2                # decode steps before the timed one: the second is captured as a graph

# ------------------------------------------------------------------------------- models
_LLAMA3 = {
    "architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": 32, "hidden_size": 4096,
    "num_attention_heads": 32, "num_key_value_heads": 8, "head_dim": 128, "intermediate_size": 14336,
    "vocab_size": 128256, "rope_theta": 500000.0, "tie_word_embeddings": False, "rms_norm_eps": 1e-5,
    "rope_scaling": {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0,
                     "original_max_position_embeddings": 8192},
    "max_position_embeddings": 8192, "hidden_act": "silu",
}


def _dirulorn() -> dict:
    dense = {"kind": "dense", "ff": 8192}
    ssm = {"type": "mamba2", "mlp": dense,
           "mixer": {"heads": 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}}
    both = {"type": "parallel", "mlp": dense,
            "mixer": {"left": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 128, "scale": 0.125,
                               "rot": {"dims": 32, "base": 500000.0,
                                       "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}},
                      "right": {"width": 2560, "blocks": 10, "conv": 4}}}
    return {"architecture": "Dirulorn", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5},
            "layers": [both if i % 2 else ssm for i in range(16)]}


def _vovalix() -> dict:
    moe = {"kind": "moe", "expert": {"ff": 2048, "limit": 7.0}, "shared": {"ff": 2048, "limit": 7.0},
           "router": {"experts": 32, "top": 4, "groups": {"count": 8, "keep": 4}}}
    attention = {"type": "attention", "mlp": moe,
                 "mixer": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": 1024}}}
    gla = {"type": "gla", "mlp": moe, "mixer": {"heads": 16, "dim": 64, "vdim": 128, "tau": 8.0, "rank": 32}}
    delta = {"type": "delta", "mlp": moe, "mixer": {"heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "conv": 4}}
    return {"architecture": "Vovalix", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5}, "logit_scale": 1.0,
            "layers": [(attention, gla, delta, gla)[i % 4] for i in range(16)]}


def _tazunex() -> dict:
    dense = {"kind": "dense", "ff": 8192}
    attention = {"type": "attention", "mlp": dense,
                 "mixer": {"heads": 32, "kv_heads": 8, "dim": 64, "vdim": 64, "scale": 0.125, "mask": {"size": 1024},
                           "rot": {"dims": 64, "base": 500000.0}}}
    latent = {"type": "latent_attention", "mlp": dense,
              "mixer": {"heads": 16, "dim": 128, "rot_dim": 32, "vdim": 128, "kv_rank": 96, "q_rank": 1024,
                        "scale": 0.1, "mask": {"size": 1024}, "rot": {"dims": 32, "base": 500000.0}}}
    memory = {"type": "mlstm", "mlp": dense, "mixer": {"heads": 16, "dim": 64, "vdim": 128, "gate_cap": 15.0}}
    return {"architecture": "Tazunex", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5}, "logit_softcap": 30.0,
            "layers": [(attention, memory, latent, memory)[i % 4] for i in range(16)]}


def _sopulorn() -> dict:
    dense = {"kind": "dense", "ff": 8192, "limit": 7.0}
    moe = {"kind": "moe", "expert": {"ff": 2048}, "router": {"experts": 32, "top": 4}, "shared": {"ff": 2048}}
    mixer = {"heads": 16, "kv_heads": 4, "dim": 128, "vdim": 64, "scale": 0.09, "rot": {"dims": 128, "base": 500000.0}}
    return {"architecture": "Sopulorn", "vocab": 32000, "width": 2048, "norm": {"eps": 1e-5},
            "embedding": {"bigram": {"buckets": 60013, "mul_prev": 8191, "mul_cur": 131}},
            "layers": [{"type": "attention", "mixer": dict(mixer, kv_from=7) if i >= 8 else mixer,
                        "mlp": moe if i else dense} for i in range(16)]}


CONFIGS = {
    "llama-8b": _LLAMA3,
    "llama-1b": dict(_LLAMA3, num_hidden_layers=16, hidden_size=2048, head_dim=64, intermediate_size=8192,
                     rope_scaling=dict(_LLAMA3["rope_scaling"], factor=32.0), tie_word_embeddings=True),
    "dirulorn": _dirulorn(), "vovalix": _vovalix(), "tazunex": _tazunex(), "sopulorn": _sopulorn(),
}
ROUTED = ("vovalix", "sopulorn")
TIED = ("llama-1b", "vovalix", "tazunex")


def _vocab(config: dict) -> int:
    return config["vocab"] if "vocab" in config else config["vocab_size"]


def _width(config: dict) -> int:
    return config["width"] if "width" in config else config["hidden_size"]


def _depth(config: dict) -> int:
    return len(config["layers"]) if "layers" in config else config["num_hidden_layers"]


# -------------------------------------------------------------------------------- cases
def _case(name, model, *, dtype="bfloat16", singles=0, context=0, portions=0, portion=0, start=0, rows=1) -> dict:
    return {"name": name, "model": model, "dtype": dtype, "singles": singles, "context": context,
            "portions": portions, "portion": portion, "start": start, "rows": rows}


def listed() -> list[dict]:
    return [
        # one chat on a small model: the smallest step there is, nothing but latency
        _case("1b decode 1", "llama-1b", singles=1, context=512),
        # the headline: eight requests decode on the 8B shape; and a full batch of them
        _case("8b decode 8", "llama-8b", singles=8, context=512),
        _case("8b decode 64", "llama-8b", singles=64, context=512),
        # one long prompt at once: the largest step
        _case("8b prompt 2048", "llama-8b", portions=1, portion=2048),
        # a server under load: portions of prompts beside requests that decode
        _case("1b mixed", "llama-1b", singles=29, context=1200, portions=3, portion=512, start=512),
        # the float32 path: a short prompt, for comparisons that must not round
        _case("1b float32 prompt", "llama-1b", dtype="float32", portions=2, portion=61),
        # whole prompts of the decoders with recurrent states
        _case("dirulorn prompt 2048", "dirulorn", portions=1, portion=2048),
        _case("tazunex prompts", "tazunex", portions=2, portion=1000, rows=4),
        # prompts that are scored, several in a step: matrix states and routed experts
        _case("vovalix prompts", "vovalix", portions=3, portion=683, rows=16),
        # routed experts while decoding: few tokens, so a part of the experts, and all of them
        _case("vovalix decode 8", "vovalix", singles=8, context=512),
        _case("sopulorn decode 64", "sopulorn", singles=64, context=512),
        # a question of a few hundred tokens before routed experts
        _case("sopulorn prompt 300", "sopulorn", portions=1, portion=300, rows=32),
    ]


def _log_uniform(rng: random.Random, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng: random.Random) -> dict:
    model = rng.choice(["llama-8b", "llama-1b", "llama-1b", "dirulorn", "dirulorn", "vovalix", "vovalix", "tazunex",
                        "tazunex", "sopulorn", "sopulorn"])
    dtype = "float32" if model == "llama-1b" and rng.random() < 0.2 else "bfloat16"
    most = 120 if dtype == "float32" else 2048
    kind = rng.choice(["decode", "prompt", "mixed"])
    singles = context = portions = portion = start = 0
    if kind != "prompt":
        singles = _log_uniform(rng, 1, 16 if dtype == "float32" else 64)
        context = _log_uniform(rng, 48, 1500 if singles <= 32 else 700)
    if kind != "decode":
        portions = _log_uniform(rng, 1, 4)
        portion = _log_uniform(rng, 16, (most - singles) // portions)
        start = rng.choice([0, 0, _log_uniform(rng, 16, 1200)])
    case = _case("", model, dtype=dtype, singles=singles, context=context, portions=portions, portion=portion,
                 start=start, rows=min(portion, 16) if model in ROUTED and portions else 1)
    del case["name"]
    return case


def _contexts(case: dict) -> list[int]:
    return [max(WARM + 1, case["context"] - (i * 37) % (case["context"] // 4 + 1)) for i in range(case["singles"])]


def _portions(case: dict) -> list[int]:
    return [case["portion"] - (i * 29) % (case["portion"] // 8 + 1) for i in range(case["portions"])]


def _wanted(case: dict, length: int) -> list[int]:
    n = min(case["rows"], length)
    return [(i + 1) * length // n - 1 for i in range(n)]


def _sequences(case: dict, seed: int) -> list[tuple[list[int], int]]:
    """Every request's tokens and how many of them were run before the step: decoding requests first."""
    rng = random.Random(seed * 7919 + 17)
    vocab = _vocab(CONFIGS[case["model"]])
    sizes = [(n, 1) for n in _contexts(case)] + [(case["start"], n) for n in _portions(case)]
    return [([rng.randrange(vocab) for _ in range(before + now)], before) for before, now in sizes]


# ------------------------------------------------------------------------------ weights
def _weight(model: str, seed: int, name: str, shape, generator: torch.Generator) -> torch.Tensor:
    """float32 values of a checkpoint's tensor, all of them numbers that bfloat16 holds."""
    config = CONFIGS[model]
    stream = _width(config) ** -0.5 if model in TIED else 1.0     # rms of the embedded rows
    # what one sublayer adds to them; less before routers, where a near-tie of two experts turns into another row
    small = (0.2 if model in ROUTED else 0.5) * stream / math.sqrt(2 * _depth(config))
    generator.manual_seed((seed << 32 | zlib.crc32(name.encode())) & (2 ** 62 - 1))
    out = torch.empty(tuple(shape), dtype=torch.float32, device=DEVICE)
    last = name[:-len(".weight")] if name.endswith(".weight") else name
    last, inner = last.rsplit(".", 1)[-1], last.rsplit(".", 1)[0].rsplit(".", 1)[-1]
    if last in ("A_log", "dt_bias", "lam") or (last == "b" and inner == "f"):
        out.uniform_(0.0, 1.0, generator=generator)
        if last == "A_log":
            out = torch.log(1.0 + 15.0 * out)                     # rates of 1 to 16
        elif last == "dt_bias":
            out = torch.log(torch.expm1(torch.exp(out * math.log(100.0)) * 0.001))  # steps of 0.001 to 0.1
        elif last == "lam":
            out = torch.log(torch.expm1(0.0005 + 0.025 * out))    # decays of 0.9 to 0.998 at a half-open gate
        else:
            out = 3.0 + 3.0 * out                                 # forget gates that start open
    else:
        out.normal_(generator=generator)
        post = last in ("norm1b", "norm2b") or (last == "out" and inner in ("left", "right"))
        if post:                                                  # gain of a norm behind a sublayer
            out.mul_(0.1 * small).add_(small - (1.0 if model == "sopulorn" else 0.0))
        elif "norm" in last:
            offset = model in ROUTED and (last in ("norm1", "norm2") or inner == "final")
            out.mul_(0.1).add_(0.0 if offset else 1.0)
        elif last == "D":
            out.mul_(0.1).add_(1.0)
        elif last == "b":
            out.mul_(1.0 if inner in ("i", "a2") else 0.1).add_({"i": -4.0, "a2": 2.0}.get(inner, 0.0))
        elif last == "sink":
            pass
        elif last in ("embed", "embed_tokens", "bigram"):
            out.mul_(stream * (0.5 ** 0.5 if model == "sopulorn" else 1.0))
        else:
            out.mul_(shape[-1] ** -0.5)
            normed = model in ("tazunex", "sopulorn") or (model == "dirulorn" and inner in ("left", "right"))
            if last in ("o", "o_proj", "down", "down_proj") and not normed:
                out.mul_(2.0 * small)
    return out.to(torch.bfloat16).float()


# -------------------------------------------------------------------------- preparation
class _State:
    def __init__(self, runner, manager, entries) -> None:
        self.runner, self.manager, self.entries = runner, manager, entries


def prepare(case: dict, seed: int) -> _State:
    from kvcore_amd.cache.kv_manager import KVManager, plan_groups
    from kvcore_amd.engine.runner import ModelRunner, StepEntry, build_model

    dtype = getattr(torch, case["dtype"])
    model = build_model(".", dtype, DEVICE, load_format="random", seed=seed, config_override=CONFIGS[case["model"]],
                        pack_weights=False)
    generator = torch.Generator(device=DEVICE)
    for name, (bound, row, rows) in model.checkpoint_map().items():
        place = bound.tensor.narrow(0, row, rows)
        place.copy_(_weight(case["model"], seed, name, place.shape, generator))
    model.weights_loaded()
    model.pack_product_weights()

    sequences = _sequences(case, seed)
    step_tokens = sum(len(tokens) - before for tokens, before in sequences)
    most = max(step_tokens, FILL)
    seqs = len(sequences)
    pages = sum(-(-len(tokens) // PAGE) for tokens, _ in sequences) + 1
    groups = plan_groups([g.need for g in model.cache_groups], PAGE, pages)
    manager = KVManager(groups, max_num_seqs=seqs, max_model_len=MAX_LEN)
    runner = ModelRunner(model, page_size=[g.page_size for g in groups], num_pages=[g.num_pages for g in groups],
                         max_num_seqs=seqs, max_num_tokens=most, max_model_len=MAX_LEN)

    def entry(r: int, first: int, last: int, want=(), name="") -> StepEntry:
        rid = f"{name}{r}"
        if not manager.is_admitted(rid):
            manager.admit(rid)
            runner.forget(manager.slot_of(rid))
        if manager.allocate(rid, first, last - first) is None:
            raise RuntimeError("the pages do not suffice")
        return StepEntry(rid, manager.slot_of(rid), first, sequences[r][0][first:last], manager.page_ids(rid),
                         want, manager.released_counts(rid))

    # a step of these portions on requests that then leave, as an engine's profile step does: its
    # buffers are there before the step that counts
    if case["portions"]:
        short = [(r, len(tokens) - before) for r, (tokens, before) in enumerate(sequences)]
        runner.step([entry(r, 0, n, tuple(_wanted(case, n)) if n > 1 else (0,), "warm") for r, n in short])
        for r, _ in short:
            runner.forget(manager.slot_of(f"warm{r}"))
            manager.free(f"warm{r}")

    decode_only = not case["portions"]
    done = [0] * seqs
    until = [before - WARM if decode_only else before for _, before in sequences]
    while any(done[r] < until[r] for r in range(seqs)):
        left, batch = most, []
        for r in range(seqs):
            n = min(until[r] - done[r], left)
            if n > 0:
                batch.append((r, n))
                left -= n
        runner.step([entry(r, done[r], done[r] + n) for r, n in batch])
        for r, n in batch:
            done[r] += n
            manager.release_behind_window(str(r), done[r])
    for _ in range(WARM if decode_only else 0):
        runner.step([entry(r, done[r], done[r] + 1, (0,)) for r in range(seqs)])
        for r in range(seqs):
            done[r] += 1
            manager.release_behind_window(str(r), done[r])
    entries = []
    for r, (tokens, before) in enumerate(sequences):
        now = len(tokens) - before
        entries.append(entry(r, before, len(tokens), tuple(_wanted(case, now)) if r >= case["singles"] else (0,)))
    return _State(runner, manager, entries)


def run(state: _State) -> dict:
    """The step: the wanted logits, and the recurrent states that it leaves."""
    out = state.runner.step(state.entries)
    return {"logits": out.logits, "states": list(state.runner.states)}


# --------------------------------------------------------------------------------- work
def work(case: dict) -> dict:
    """Every weight that the step's tokens need once, the cached keys and values and the states once;
    two operations per weight and token, four per visible key and element of a head, and those of the states."""
    from kvcore_amd.registry import resolve_architecture
    from kvcore_amd.weights.loader import checkpoint_layout

    config = CONFIGS[case["model"]]
    arch = resolve_architecture(config)
    layout = checkpoint_layout(arch.build_spec(arch.parse_config(config)))
    spans = [(n, 1) for n in _contexts(case)] + [(case["start"], n) for n in _portions(case)]
    tokens = sum(n for _, n in spans)
    wanted = case["singles"] + sum(len(_wanted(case, n)) for n in _portions(case))
    size = 4 if case["dtype"] == "float32" else 2
    moved = flops = 0.0
    for name, (shape, _, _) in layout.items():
        count = math.prod(shape)
        table = name.rsplit(".weight", 1)[0] in ("embed", "model.embed_tokens", "bigram", "head", "lm_head")
        if table:
            if name.startswith(("head", "lm_head")) or (case["model"] in TIED and "embed" in name):
                moved += count * size
                flops += 2.0 * count * wanted
            else:
                moved += tokens * shape[-1] * size
        elif ".mlp.e" in name:
            router = config["layers"][int(name[1:name.index(".")])]["mlp"]["router"]
            share = router["top"] / router["experts"]
            moved += count * size * (1.0 - (1.0 - share) ** tokens)
            flops += 2.0 * count * tokens * share
        else:
            moved += count * size
            flops += 2.0 * count * tokens

    def attend(heads, kv_elems, dim, window=None, chunk=None):
        nonlocal moved, flops
        for before, now in spans:
            pairs = held = 0
            for p in (before, before + now - 1):
                seen = p + 1 if not window else min(p + 1, window)
                pairs += (seen if not chunk else p % chunk + 1) * now / 2
                held = max(held, seen if not chunk else p % chunk + 1)
            flops += 2.0 * pairs * heads * dim
            moved += (max(held, now) + now) * kv_elems * size

    def state(elems, ops):
        nonlocal moved, flops
        moved += 8.0 * elems * len(spans)
        flops += float(ops) * elems * tokens

    if "layers" not in config:
        for _ in range(_depth(config)):
            d = config["head_dim"]
            attend(config["num_attention_heads"], 2 * config["num_key_value_heads"] * d, 2 * d)
    for layer in config.get("layers", ()):
        m = layer["mixer"]
        kind = layer["type"]
        mask = (m.get("mask") or {}).get("size")
        if kind == "parallel":
            left = m["left"]
            attend(left["heads"], left["kv_heads"] * (left["dim"] + left["vdim"]), left["dim"] + left["vdim"])
            state(m["right"]["width"], 6)
        elif kind == "mamba2":
            state(m["heads"] * m["vdim"] * m["state"], 5)
        elif kind in ("gla", "mlstm", "delta"):
            state(m["heads"] * m["dim"] * m["vdim"], 8 if kind == "delta" else 5)
        elif kind == "latent_attention":
            attend(m["heads"], m["kv_rank"] + m["rot_dim"], 2 * m["kv_rank"] + m["rot_dim"], window=mask)
        else:
            chunk = mask if case["model"] == "vovalix" else None
            attend(m["heads"], m["kv_heads"] * (m["dim"] + m["vdim"]), m["dim"] + m["vdim"],
                   window=None if chunk else mask, chunk=chunk)
    return {"bytes": moved, "flops": flops}


def tolerance(case: dict) -> dict:
    """About four times the error against 64 bits: 1.2e-6 in float32; in bfloat16 0.0025 for Llama's logits and
    0.0033 for the recurrent decoders', whose states of deep layers carry more; routed experts add their near-ties."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 2e-4}
    if case["model"].startswith("llama"):
        return {"rel": 0.012, "max": 0.3}
    return {"rel": 0.03 if case["model"] in ROUTED else 0.02, "max": 0.5}


# ------------------------------------------------------- the same in 64 bits, without the engine
class _Plain:
    """The decoders written out in float64: all tokens of all requests side by side as rows, no cache."""

    def __init__(self, model: str, seed: int, sequences: list[list[int]]) -> None:
        self.model, self.seed, self.config = model, seed, CONFIGS[model]
        self.generator = torch.Generator(device=DEVICE)
        self.lengths = [len(s) for s in sequences]
        self.tokens = torch.tensor([t for s in sequences for t in s], device=DEVICE)
        self.first = [sum(self.lengths[:i]) for i in range(len(sequences))]
        self.positions = torch.cat([torch.arange(n, device=DEVICE) for n in self.lengths]).double()
        # row of a request's token t in the side-by-side rows, padded on the right
        longest = max(self.lengths)
        self.padded = torch.tensor([[f + min(t, n - 1) for t in range(longest)]
                                    for f, n in zip(self.first, self.lengths)], device=DEVICE)
        self.alive = torch.tensor([[t < n for t in range(longest)] for n in self.lengths], device=DEVICE)
        config = self.config
        self.eps = config["norm"]["eps"] if "norm" in config else config["rms_norm_eps"]

    # ---- pieces
    def w(self, name: str, *shape: int) -> torch.Tensor:
        return _weight(self.model, self.seed, name, shape, self.generator).double()

    def product(self, x: torch.Tensor, name: str, rows: int) -> torch.Tensor:
        return x @ self.w(name, rows, x.shape[-1]).T

    def rms(self, x: torch.Tensor) -> torch.Tensor:
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + self.eps)

    def norm(self, x: torch.Tensor, name: str, offset: float = 0.0) -> torch.Tensor:
        return self.rms(x) * (self.w(name, x.shape[-1]) + offset)

    def to_time(self, x: torch.Tensor) -> torch.Tensor:
        """Rows [N, ...] -> [requests, time, ...]."""
        return x[self.padded]

    def to_rows(self, y: torch.Tensor) -> torch.Tensor:
        return y[self.alive]

    def rotate(self, x: torch.Tensor, dims: int, frequencies: torch.Tensor, interleaved: bool) -> torch.Tensor:
        angle = self.positions[:, None, None] * frequencies
        c, s = torch.cos(angle), torch.sin(angle)
        out = x.clone()
        a, b = ((slice(0, dims, 2), slice(1, dims, 2)) if interleaved
                else (slice(0, dims // 2), slice(dims // 2, dims)))
        u, v = x[..., a], x[..., b]
        out[..., a], out[..., b] = u * c - v * s, v * c + u * s
        return out

    def frequencies(self, dims: int, base: float, factor=None, low=1.0, high=4.0, original=8192) -> torch.Tensor:
        f = base ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device=DEVICE) / dims)
        if factor:
            turns = original * f / (2 * math.pi)
            blend = ((turns - low) / (high - low)).clamp(0.0, 1.0)
            f = f / factor * (1.0 - blend) + f * blend
        return f

    def attend(self, q, k, v, scale, *, window=None, chunk=None, slopes=None, sink=None) -> torch.Tensor:
        """``q [N, heads, d]``, ``k, v [N, kv_heads, ..]``; ``sink [heads]``: a score without a value."""
        rep = q.shape[1] // k.shape[1]
        out = torch.empty(*q.shape[:2], v.shape[-1], dtype=q.dtype, device=DEVICE)
        for f, n in zip(self.first, self.lengths):
            kk = k[f:f + n].repeat_interleave(rep, 1).permute(1, 2, 0).contiguous()
            vv = v[f:f + n].repeat_interleave(rep, 1).transpose(0, 1).contiguous()
            j = torch.arange(n, device=DEVICE)[None, :]
            for a in range(0, n, 512):
                b = min(n, a + 512)
                i = torch.arange(a, b, device=DEVICE)[:, None]
                scores = torch.bmm(q[f + a:f + b].transpose(0, 1).contiguous(), kk) * scale
                if slopes is not None:
                    scores -= slopes[:, None, None] * (i - j)
                hidden = j > i
                if window:
                    hidden = hidden | (i - j >= window)
                if chunk:
                    hidden = hidden | (j // chunk != i // chunk)
                scores.masked_fill_(hidden, -math.inf)
                if sink is not None:
                    scores = torch.cat([scores, sink[:, None, None].expand(-1, b - a, 1)], -1)
                weights = torch.softmax(scores, -1)
                out[f + a:f + b] = torch.bmm(weights[..., :n].contiguous(), vv).transpose(0, 1)
        return out

    def conv(self, x: torch.Tensor, taps: torch.Tensor, bias=None) -> torch.Tensor:
        y, out = self.to_time(x), 0.0
        for j in range(taps.shape[1]):
            moved = torch.nn.functional.pad(y, (0, 0, j, 0))[:, :y.shape[1]]
            out = out + moved * taps[:, taps.shape[1] - 1 - j]
        out = self.to_rows(out)
        return out if bias is None else out + bias

    def gated(self, x, p, ff, act, names=("gate", "up", "down"), suffix="") -> torch.Tensor:
        return self.product(act(self.product(x, f"{p}.{names[0]}{suffix}", ff), self.product(x, f"{p}.{names[1]}{suffix}", ff)),
                            f"{p}.{names[2]}{suffix}", x.shape[-1])

    def routed(self, x, p, choice, weight, experts, ff, act) -> torch.Tensor:
        out = torch.zeros_like(x)
        for e in range(experts):
            rows, place = torch.nonzero(choice == e, as_tuple=True)
            if rows.numel():
                out[rows] += weight[rows, place][:, None] * self.gated(x[rows], f"{p}.e{e}", ff, act)
        return out

    # ---- decoders: rows [N, width] in front of the head
    def llama(self) -> torch.Tensor:
        c = self.config
        H, heads, kv, d, ff = (c["hidden_size"], c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"],
                               c["intermediate_size"])
        s = c["rope_scaling"]
        freq = self.frequencies(d, c["rope_theta"], s["factor"], s["low_freq_factor"], s["high_freq_factor"],
                                s["original_max_position_embeddings"])
        x = self.w("model.embed_tokens.weight", c["vocab_size"], H)[self.tokens]
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}"
            h = self.norm(x, f"{p}.input_layernorm.weight")
            q, k, v = (self.product(h, f"{p}.self_attn.{n}_proj.weight", m * d).view(-1, m, d)
                       for n, m in (("q", heads), ("k", kv), ("v", kv)))
            o = self.attend(self.rotate(q, d, freq, False), self.rotate(k, d, freq, False), v, d ** -0.5)
            x = x + self.product(o.flatten(1), f"{p}.self_attn.o_proj.weight", H)
            h = self.norm(x, f"{p}.post_attention_layernorm.weight")
            x = x + self.gated(h, f"{p}.mlp", ff, _silu_mul, ("gate_proj", "up_proj", "down_proj"), ".weight")
        return self.norm(x, "model.norm.weight")

    def layer_norm(self, x: torch.Tensor, name: str) -> torch.Tensor:
        return torch.nn.functional.layer_norm(x, x.shape[-1:], self.w(name, x.shape[-1]),
                                              self.w(name + ".b", x.shape[-1]), self.eps)

    def dirulorn(self) -> torch.Tensor:
        c = self.config
        x = self.w("embed", c["vocab"], c["width"])[self.tokens]
        for i, layer in enumerate(c["layers"]):
            h = self.layer_norm(x, f"l{i}.norm1")
            x = x + getattr(self, layer["type"])(h, f"l{i}.mix", layer["mixer"])
            x = x + self.gated(self.layer_norm(x, f"l{i}.norm2"), f"l{i}.mlp", layer["mlp"]["ff"], _silu_mul)
        return self.layer_norm(x, "final.norm")

    def mamba2(self, h, p, m) -> torch.Tensor:
        nh, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        inner, conv = nh * P, nh * P + 2 * G * N
        z, xbc, dt = self.product(h, p + ".in", inner + conv + nh).split([inner, conv, nh], -1)
        xbc = _silu(self.conv(xbc, self.w(p + ".conv", conv, m["conv"]), self.w(p + ".conv.b", conv)))
        x, B, C = xbc.split([inner, G * N, G * N], -1)
        x = x.reshape(-1, nh, P)
        B, C = (y.reshape(-1, G, N).repeat_interleave(nh // G, 1) for y in (B, C))
        dt = _softplus(dt + self.w(p + ".dt_bias", nh))
        decay = torch.exp(-torch.exp(self.w(p + ".A_log", nh)) * dt)
        y = self.scan(C, B, x * dt[..., None], decay[..., None]) + self.w(p + ".D", nh)[:, None] * x
        y = (y.flatten(1) * _silu(z)).view(-1, m["norm_groups"], inner // m["norm_groups"])
        return self.product(self.rms(y).flatten(1) * self.w(p + ".norm", inner), p + ".o", h.shape[-1])

    def scan(self, q, k, v, decay, beta=None) -> torch.Tensor:
        """``q, k [N, heads, d]``, ``v [N, heads, dv]``, ``decay [N, heads, d or 1]``: a matrix state a head
        that shrinks and takes ``k v^T`` (with ``beta [N, heads]`` the part of v that it does not answer yet)."""
        q, k, v, decay = (self.to_time(t) for t in (q, k, v, decay))
        beta = None if beta is None else self.to_time(beta)
        R, T, heads, d = q.shape
        S = torch.zeros(R, heads, d, v.shape[-1], dtype=q.dtype, device=DEVICE)
        out = torch.empty(R, T, heads, v.shape[-1], dtype=q.dtype, device=DEVICE)
        for t in range(T):
            S *= decay[:, t, :, :, None]
            u = v[:, t]
            if beta is not None:
                u = beta[:, t, :, None] * (u - (S * k[:, t, :, :, None]).sum(2))
            S.addcmul_(k[:, t, :, :, None], u[:, :, None, :])
            out[:, t] = (S * q[:, t, :, :, None]).sum(2)
        return self.to_rows(out)

    def parallel(self, h, p, m) -> torch.Tensor:
        a, b, H = m["left"], m["right"], h.shape[-1]
        rot = a["rot"]
        freq = self.frequencies(rot["dims"], rot["base"], **rot["scaling"])
        q = self.product(h, p + ".left.q", a["heads"] * a["dim"]).view(-1, a["heads"], a["dim"])
        k = self.product(h, p + ".left.k", a["kv_heads"] * a["dim"]).view(-1, a["kv_heads"], a["dim"])
        v = self.product(h, p + ".left.v", a["kv_heads"] * a["vdim"]).view(-1, a["kv_heads"], a["vdim"])
        q, k = (self.rotate(self.norm(y, f"{p}.left.{n}.norm"), rot["dims"], freq, True) for y, n in ((q, "q"), (k, "k")))
        left = self.product(self.attend(q, k, v, a["scale"]).flatten(1), p + ".left.o", H)
        W, nb = b["width"], b["blocks"]
        r = p + ".right"
        y = torch.nn.functional.gelu(self.product(h, r + ".y", W) + self.w(r + ".y.b", W), approximate="tanh")
        u = self.conv(self.product(h, r + ".x", W) + self.w(r + ".x.b", W), self.w(r + ".conv", W, b["conv"]),
                      self.w(r + ".conv.b", W))
        ub = u.view(-1, nb, W // nb).transpose(0, 1).contiguous()
        ga, gi = (torch.sigmoid(torch.bmm(ub, self.w(f"{r}.{n}", nb, W // nb, W // nb).transpose(1, 2).contiguous())
                                .transpose(0, 1) + self.w(f"{r}.{n}.b", nb, W // nb)).reshape(-1, W) for n in ("ra", "ri"))
        a_t = torch.exp(-8.0 * ga * _softplus(self.w(r + ".lam", W)))
        drive, decay = self.to_time(torch.sqrt(1.0 - a_t * a_t) * gi * u), self.to_time(a_t)
        S, out = torch.zeros_like(drive[:, 0]), torch.empty_like(drive)
        for t in range(drive.shape[1]):
            S = decay[:, t] * S + drive[:, t]
            out[:, t] = S
        right = self.product(self.to_rows(out) * y, r + ".o", H)
        return 0.5 * (self.norm(left, p + ".left.out") + self.norm(right, p + ".right.out"))

    def vovalix(self) -> torch.Tensor:
        c = self.config
        x = self.w("embed", c["vocab"], c["width"])[self.tokens]
        for i, layer in enumerate(c["layers"]):
            h = self.norm(x, f"l{i}.norm1", 1.0)
            p, r = f"l{i}.mlp", layer["mlp"]["router"]
            per = r["experts"] // r["groups"]["count"]
            scores = torch.softmax(self.product(h, p + ".router", r["experts"]), -1)
            kept = scores.view(-1, r["groups"]["count"], per).amax(-1).topk(r["groups"]["keep"], -1).indices
            mask = torch.zeros(h.shape[0], r["groups"]["count"], dtype=torch.bool, device=DEVICE).scatter_(1, kept, True)
            best = scores.masked_fill(~mask.repeat_interleave(per, 1), -1.0).topk(r["top"], -1)
            weight = best.values / best.values.sum(-1, keepdim=True)
            ff = layer["mlp"]["expert"]["ff"]
            y = self.routed(h, p, best.indices, weight, r["experts"], ff, _clamped)
            y = y + self.gated(h, p + ".shared", layer["mlp"]["shared"]["ff"], _clamped)
            x = x + y + getattr(self, "vovalix_" + layer["type"])(h, f"l{i}.mix", layer["mixer"])
        return self.norm(x, "final.norm", 1.0)

    def heads(self, h, p, name, heads, dim) -> torch.Tensor:
        return self.product(h, f"{p}.{name}", heads * dim).view(-1, heads, dim)

    def vovalix_attention(self, h, p, m) -> torch.Tensor:
        H, G = m["heads"], m["kv_heads"]
        q, k = self.rms(self.heads(h, p, "q", H, m["dim"])), self.rms(self.heads(h, p, "k", G, m["dim"]))
        slopes = 2.0 ** (-8.0 * torch.arange(1, H + 1, dtype=torch.float64, device=DEVICE) / H)
        o = self.attend(q, k, self.heads(h, p, "v", G, m["vdim"]), m["scale"], chunk=m["mask"]["size"], slopes=slopes)
        return self.product(o.flatten(1), p + ".o", h.shape[-1])

    def head_gate(self, o, h, p, m) -> torch.Tensor:
        inner = m["heads"] * m["vdim"]
        y = self.norm(o, p + ".norm").flatten(1) * _silu(self.product(h, p + ".g", inner))
        return self.product(y, p + ".o", h.shape[-1])

    def vovalix_gla(self, h, p, m) -> torch.Tensor:
        H, d = m["heads"], m["dim"]
        z = self.product(self.product(h, p + ".a1", m["rank"]), p + ".a2", H * d) + self.w(p + ".a2.b", H * d)
        decay = torch.sigmoid(z).pow(1.0 / m["tau"]).view(-1, H, d)
        o = self.scan(self.heads(h, p, "q", H, d) * d ** -0.5, self.heads(h, p, "k", H, d),
                      self.heads(h, p, "v", H, m["vdim"]), decay)
        return self.head_gate(o, h, p, m)

    def vovalix_delta(self, h, p, m) -> torch.Tensor:
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (_silu(self.conv(self.product(h, f"{p}.{n}", r), self.w(f"{p}.{n}.conv", r, m["conv"])))
                   for n, r in (("q", G * d), ("k", G * d), ("v", H * dv)))
        q, k = (y.view(-1, G, d) for y in (q, k))
        q, k = (y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
        q, k = (y.repeat_interleave(H // G, 1) for y in (q * d ** -0.5, k))
        beta = torch.sigmoid(self.product(h, p + ".b", H))
        g = torch.exp(-torch.exp(self.w(p + ".A_log", H)) * _softplus(self.product(h, p + ".a", H) + self.w(p + ".dt_bias", H)))
        return self.head_gate(self.scan(q, k, v.view(-1, H, dv), g[..., None], beta), h, p, m)

    def tazunex(self) -> torch.Tensor:
        c = self.config
        x = self.w("embed", c["vocab"], c["width"])[self.tokens]
        for i, layer in enumerate(c["layers"]):
            y = getattr(self, "tazunex_" + layer["type"])(self.norm(x, f"l{i}.norm1"), f"l{i}.mix", layer["mixer"])
            x = x + self.norm(y, f"l{i}.norm1b")
            y = self.gated(self.norm(x, f"l{i}.norm2"), f"l{i}.mlp", layer["mlp"]["ff"], _gelu_mul)
            x = x + self.norm(y, f"l{i}.norm2b")
        return self.norm(x, "final.norm")

    def tazunex_attention(self, h, p, m) -> torch.Tensor:
        H, G, d, rot = m["heads"], m["kv_heads"], m["dim"], m["rot"]
        freq = self.frequencies(rot["dims"], rot["base"])
        q, raw = self.product(h, p + ".q", H * d), self.product(h, p + ".k", G * d)
        q, k = (self.rotate(self.norm(y, f"{p}.{n}.norm").view(-1, r, d), rot["dims"], freq, False)
                for y, n, r in ((q, "q", H), (raw, "k", G)))
        o = self.attend(q, k, raw.view(-1, G, d), m["scale"], window=m["mask"]["size"], sink=self.w(p + ".sink", H))
        return self.product(o.flatten(1), p + ".o", h.shape[-1])

    def tazunex_latent_attention(self, h, p, m) -> torch.Tensor:
        H, d, r, rank = m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
        freq = self.frequencies(r, m["rot"]["base"])
        q = self.heads(self.norm(self.product(h, p + ".dq", m["q_rank"]), p + ".dq.norm"), p, "uq", H, d + r)
        down = self.product(h, p + ".dkv", rank + r)
        latent = self.norm(down[:, :rank], p + ".dkv.norm")
        turned = self.rotate(down[:, rank:].reshape(-1, 1, r), r, freq, True).expand(-1, H, -1)
        q = torch.cat([q[..., :d], self.rotate(q[..., d:], r, freq, True)], -1)
        k = torch.cat([self.heads(latent, p, "uk", H, d), turned], -1)
        o = self.attend(q, k, self.heads(latent, p, "uv", H, m["vdim"]), m["scale"], window=m["mask"]["size"])
        gate = torch.sigmoid(self.product(h, p + ".g", H))
        return self.product((o * gate[..., None]).flatten(1), p + ".o", h.shape[-1])

    def tazunex_mlstm(self, h, p, m) -> torch.Tensor:
        H, d, dv, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k = self.heads(h, p, "q", H, d) * d ** -0.5, self.heads(h, p, "k", H, d)
        gi, gf = (cap * torch.tanh((self.product(h, f"{p}.{n}", H) + self.w(f"{p}.{n}.b", H)) / cap) for n in ("i", "f"))
        gi, gf = self.to_time(gi), self.to_time(torch.nn.functional.logsigmoid(gf))
        top, keep, take, tops = torch.zeros_like(gi[:, 0]), torch.empty_like(gi), torch.empty_like(gi), torch.empty_like(gi)
        for t in range(gi.shape[1]):
            new = torch.maximum(gf[:, t] + top, gi[:, t])
            keep[:, t], take[:, t], tops[:, t] = torch.exp(gf[:, t] + top - new), torch.exp(gi[:, t] - new), new
            top = new
        keep, take, tops = (self.to_rows(y) for y in (keep, take, tops))
        v = torch.cat([self.heads(h, p, "v", H, dv), torch.ones(h.shape[0], H, 1, dtype=h.dtype, device=DEVICE)], -1)
        o = self.scan(q, k * take[..., None], v, keep[..., None])  # the last column is the memory's normaliser
        o = o[..., :dv] / (torch.maximum(o[..., dv].abs(), torch.exp(-tops)) + 1e-6)[..., None]
        o = self.rms(o).flatten(1) * self.w(p + ".norm", H * dv)
        return self.product(o * torch.sigmoid(self.product(h, p + ".g", H * dv)), p + ".o", h.shape[-1])

    def sopulorn(self) -> torch.Tensor:
        c = self.config
        pair = c["embedding"]["bigram"]
        before = torch.roll(self.tokens, 1)
        row = (before * pair["mul_prev"] + self.tokens * pair["mul_cur"]) % pair["buckets"]
        row = torch.where(self.positions == 0, torch.full_like(row, pair["buckets"]), row)
        x = self.w("embed", c["vocab"], c["width"])[self.tokens] + self.w("bigram", pair["buckets"] + 1, c["width"])[row]
        held = None
        for i, layer in enumerate(c["layers"]):
            p, m, mlp = f"l{i}.mix", layer["mixer"], layer["mlp"]
            H, G, d = m["heads"], m["kv_heads"], m["dim"]
            freq = self.frequencies(m["rot"]["dims"], m["rot"]["base"])
            h = self.norm(x, f"l{i}.norm1", 1.0)

            def projected(n, heads, dim):
                return self.heads(h, p, n, heads, dim) + self.w(f"{p}.{n}.b", heads * dim).view(heads, dim)

            q = self.rotate(self.norm(projected("q", H, d), p + ".q.norm"), d, freq, False)
            if m.get("kv_from") is None:
                held = (self.rotate(self.norm(projected("k", G, d), p + ".k.norm"), d, freq, False),
                        projected("v", G, m["vdim"]))
            o = self.attend(q, *held, m["scale"], sink=torch.zeros(H, dtype=x.dtype, device=DEVICE))
            x = x + self.norm(self.product(o.flatten(1), p + ".o", c["width"]), f"l{i}.norm1b", 1.0)
            h, p = self.norm(x, f"l{i}.norm2", 1.0), f"l{i}.mlp"
            if mlp["kind"] == "dense":
                y = self.gated(h, p, mlp["ff"], _clamped)
            else:
                E = mlp["router"]["experts"]
                best = (self.product(h, p + ".router", E) + self.w(p + ".router.b", E)).topk(mlp["router"]["top"], -1)
                y = self.routed(h, p, best.indices, torch.softmax(best.values, -1), E, mlp["expert"]["ff"], _silu_mul)
                y = y + torch.sigmoid(self.product(h, p + ".shared.sg", 1)) * self.gated(
                    h, p + ".shared", mlp["shared"]["ff"], _silu_mul)
            x = x + self.norm(y, f"l{i}.norm2b", 1.0)
        return self.norm(x, "final.norm", 1.0)

    def logits(self, rows: list[int]) -> torch.Tensor:
        c = self.config
        x = getattr(self, self.model.split("-")[0])()[torch.tensor(rows, device=DEVICE)]
        if "layers" in c:
            name = "embed" if self.model in TIED else "head"
        else:
            name = "model.embed_tokens.weight" if self.model in TIED else "lm_head.weight"
        out = self.product(x, name, _vocab(c))
        cap = c.get("logit_softcap")
        return cap * torch.tanh(out / cap) if cap else out


def _silu(z):
    return z * torch.sigmoid(z)


def _softplus(z):
    return torch.logaddexp(z, torch.zeros_like(z))


def _silu_mul(g, u):
    return _silu(g) * u


def _gelu_mul(g, u):
    return torch.nn.functional.gelu(g, approximate="tanh") * u


def _clamped(g, u):
    g = g.clamp(max=7.0)
    return g * torch.sigmoid(1.702 * g) * (u.clamp(-7.0, 7.0) + 1.0)


def exact(case: dict, seed: int):
    """The wanted logits in 64 bits.  None for routed experts with a few rows only: which of two experts that
    nearly tie is chosen decides how far such a row is from its 64-bit value, not the sums' precision."""
    sequences = _sequences(case, seed)
    wanted = case["singles"] + sum(len(_wanted(case, n)) for n in _portions(case))
    if case["model"] in ROUTED and wanted < 32:
        return None
    if sum(len(t) for t, _ in sequences) > 34000:
        return None
    with torch.no_grad():
        plain = _Plain(case["model"], seed, [tokens for tokens, _ in sequences])
        rows = []
        for r, (tokens, before) in enumerate(sequences):
            want = _wanted(case, len(tokens) - before) if r >= case["singles"] else [0]
            rows += [plain.first[r] + before + i for i in want]
        return {"logits": plain.logits(rows)}
