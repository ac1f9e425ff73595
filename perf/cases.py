"""Steps of the serving engine and the exact latency quantiles, as cases whose time and outputs are measured.

A step case is one step of the engine: prompt portions of several sequences, or one more token of each, through scheduler,
staging, captured graph and LM head, the way the serving loop runs it (a step is launched, then the ids of the one before it are
read).  Models are the layers that ``bench.py --workload steps`` runs (``kvmini.harness.step_bench``: four layers at the sizes of a
1B and an 8B decoder, a vocabulary of 32768), weights and tokens are drawn from the seed.  A latency case is
``hist_quantile.batched_quantiles``, the reduction behind every report.

A pass returns the logits that were asked for and the sequences' memory as it is after the step.  Sampled ids are left out: they are
the places of the largest logits, and two of 32768 random ones are closer than bf16 tells apart in a few rows of a hundred."""

from __future__ import annotations

import math
import random
import zlib
from typing import Any, Callable, Dict, List, Optional, Tuple

import numpy as np
import torch

DEVICE = "cuda:0"
MAX_SEQS, MAX_TOKENS = 64, 2048  # of a step
DESIGNS = ("vodinex", "pipilix", "zipelix", "gebasun", "llama")
KINDS = 256  # of tokens, see _tensor
LEVELS = (0.5, 0.95, 0.99)


def _step(name: str, design: str, size: str, kind: str, seqs: int, tokens: int, weights: str = "bf16", cache: str = "bf16") -> Dict[str, Any]:
    """``tokens``: new ones of the longest sequence (kind prompt), or those it holds already when it takes one more (kind decode)."""
    return {"name": name, "design": design, "size": size, "kind": kind, "seqs": seqs, "tokens": tokens, "weights": weights, "cache": cache}


def listed() -> List[Dict[str, Any]]:
    return [
        # one chat on a small model: nothing but latency and launches
        _step("llama-1b-decode-1", "llama", "1b-layers", "decode", 1, 128),
        # the headline mix (500 requests, 20 in flight) while it decodes
        _step("llama-8b-decode-20", "llama", "8b-layers", "decode", 20, 96),
        # ... and when its short prompts arrive together, on the FP8 engine profile with an FP8 cache
        _step("llama-8b-fp8-prompts-18", "llama", "8b-layers", "prompt", 18, 15, "fp8", "fp8"),
        # a long prompt in one step: the time to its first token
        _step("llama-8b-prompt-2048", "llama", "8b-layers", "prompt", 1, 2048),
        # two conversations deep in the long-context profile
        _step("llama-8b-decode-2-long", "llama", "8b-layers", "decode", 2, 32768),
        # prompts of a few requests, ragged, on each hybrid design: chunked attention beside the delta rule,
        _step("vodinex-8b-prompts-4", "vodinex", "8b-layers", "prompt", 4, 560),
        # latent attention in a window and clamped experts,
        _step("pipilix-8b-prompts-3", "pipilix", "8b-layers", "prompt", 3, 700),
        # rotated latent attention, retention and several streams on a small model,
        _step("zipelix-1b-prompt-2048", "zipelix", "1b-layers", "prompt", 1, 2048),
        # windowed attention, state spaces and squared-relu experts
        _step("gebasun-8b-prompt-2000", "gebasun", "8b-layers", "prompt", 1, 2000),
        # the same designs while a batch decodes
        _step("zipelix-8b-decode-16", "zipelix", "8b-layers", "decode", 16, 1024),
        _step("gebasun-1b-decode-64", "gebasun", "1b-layers", "decode", 64, 1024),
        # p50 / p95 / p99 of the inter-token gaps of a fleet's run: three metrics, a few million samples each
        {"name": "latencies-3x4M", "design": "latencies", "metrics": 3, "samples": 4_000_000, "double": False},
    ]


def _between(rng: random.Random, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random) -> Dict[str, Any]:
    if rng.random() < 0.1:  # one run's 500 requests up to a fleet's
        metrics = rng.randint(1, 4)
        return {"design": "latencies", "metrics": metrics, "samples": _between(rng, 500, 12_000_000 // metrics), "double": rng.random() < 0.5}
    design = rng.choice(DESIGNS + ("llama",))
    size = rng.choice(("1b-layers", "8b-layers"))
    weights = cache = "bf16"
    if design == "llama":
        weights, cache = rng.choice(("bf16", "bf16", "fp8", "mxfp4")), rng.choice(("bf16", "bf16", "fp8"))
    if rng.random() < 0.55:
        seqs = _between(rng, 1, 32)
        tokens = _between(rng, min(12, MAX_TOKENS // seqs), MAX_TOKENS // seqs)
        kind = "prompt"
    else:
        seqs = _between(rng, 1, MAX_SEQS)
        tokens = _between(rng, 16, min(65536 // seqs, 32768 if design == "llama" else 4096))
        kind = "decode"
    c = _step("", design, size, kind, seqs, max(2, tokens), weights, cache)
    del c["name"]
    return c


# ---- what a case consists of ---------------------------------------------------------------------------------------
def _config(case: Dict[str, Any]) -> Any:
    from kvmini.harness.step_bench import configs

    return configs(case["size"])[DESIGNS.index(case["design"])]


def _lengths(case: Dict[str, Any]) -> List[int]:
    """``tokens`` of every sequence: ragged, the longest first, the shortest a quarter less."""
    n = case["tokens"]
    return [n - (37 * i) % (n // 4 + 1) for i in range(case["seqs"])]


def _tokens(case: Dict[str, Any], seed: int, vocab: int) -> List[List[int]]:
    """Every sequence's tokens, those of this step at the end."""
    r = np.random.default_rng([seed, 11])
    extra = 1 if case["kind"] == "decode" else 0
    return [r.integers(0, vocab, n + extra).tolist() for n in _lengths(case)]


def _wanted(case: Dict[str, Any], n: int) -> List[int]:
    """Places in a portion of ``n`` tokens whose logits are asked for: the last ones, 64 rows of a step, which the LM head serves anyway."""
    return list(range(max(0, n - max(1, MAX_SEQS // case["seqs"])), n))


def _generator(seed: int, name: str) -> torch.Generator:
    g = torch.Generator(device=DEVICE)
    g.manual_seed((seed * 1_000_003 + zlib.crc32(name.encode())) & 0x7FFFFFFF)
    return g


def _normal(seed: int, name: str, shape: Tuple[int, ...]) -> torch.Tensor:
    return torch.randn(shape, generator=_generator(seed, name), device=DEVICE, dtype=torch.float32)


def _kinds(seed: int, width: int) -> torch.Tensor:
    return torch.sign(_normal(seed, "kinds", (KINDS, width)))


def _experts_of(seed: int, experts: int, top: int) -> torch.Tensor:
    return torch.rand((KINDS, experts), generator=_generator(seed, f"experts {experts}"), device=DEVICE).topk(top, dim=1).indices


def _tensor(seed: int, name: str, shape: Tuple[int, ...], moe: Any = None, tied: bool = False) -> torch.Tensor:
    """A weight of a checkpoint, bf16: matrices have variance 1 / fan-in, the rest is spread around its neutral value.

    Tokens are of one of 256 kinds, a direction in their embeddings, and routers send a kind to experts of its own: like a trained
    router's and unlike a random one's, its choices are clear ones that rounding does not turn, spread evenly over the experts."""
    leaf = name.rsplit(".", 1)[-1]
    r = _normal(seed, name, shape)
    if name == "embed":
        r = (r + _kinds(seed, shape[1])[torch.arange(shape[0], device=DEVICE) % KINDS]) / math.sqrt(2.0)
        r = r / math.sqrt(shape[1]) if tied else r
    elif leaf == "router":
        at = _experts_of(seed, moe.experts, moe.top)
        chosen = torch.zeros((KINDS, moe.experts), device=DEVICE).scatter_(1, at, 1.0)
        r = r / math.sqrt(shape[1]) / 16 + chosen.T @ _kinds(seed, shape[1]) * (6.0 / shape[1])
    elif leaf.startswith("norm"):
        r = 1.0 + 0.1 * r
    elif leaf == "conv":
        r = r / math.sqrt(shape[1])
    elif leaf in ("in", "out", "mix") and ".hc" in name:
        r = 0.1 * r + (1.0 / shape[0] if leaf == "in" else 1.0 if leaf == "out" else torch.eye(shape[0], device=DEVICE))
    elif leaf == "correction":
        r = 0.01 * r
    elif leaf in ("D", "sink", "rel"):
        pass
    elif leaf == "b" and len(shape) == 1:
        r = 0.1 * r
    elif leaf in ("A_log", "dt_bias"):
        r = r - 1.0
    else:
        r = r / math.sqrt(shape[-1])
    return r.to(torch.bfloat16)


def _llama_shapes(cfg: Any) -> Dict[str, Tuple[int, int]]:
    w, q, kv, ff = cfg.hidden_size, cfg.num_heads * cfg.head_dim, cfg.num_kv_heads * cfg.head_dim, cfg.intermediate_size
    return {"q": (q, w), "k": (kv, w), "v": (kv, w), "o": (w, q), "gate": (ff, w), "up": (ff, w), "down": (w, ff)}


def _checkpoint(cfg: Any, seed: int) -> Callable[[str], torch.Tensor]:
    """``get(name)`` of a seed's weights."""
    if hasattr(cfg, "intermediate_size"):
        shapes = {f"l{i}.{n}": s for i in range(cfg.num_layers) for n, s in _llama_shapes(cfg).items()}
        shapes.update({"embed": (cfg.vocab_size, cfg.hidden_size), "head": (cfg.vocab_size, cfg.hidden_size)})
        return lambda name: _tensor(seed, name, shapes[name])
    from kvmini.models.hybrid import tensor_shapes

    every = tensor_shapes(cfg)
    layer = lambda name: cfg.layers[int(name[1 : name.index(".")])].moe if name.endswith(".router") else None  # noqa: E731
    return lambda name: _tensor(seed, name, every[name], layer(name), cfg.tied_head)


def _weights(cfg: Any, get: Callable[[str], torch.Tensor]) -> Any:
    if not hasattr(cfg, "intermediate_size"):
        from kvmini.models.hybrid import build_weights
        from kvmini.ops.hip_mixers import layout

        return build_weights(cfg, get, torch.bfloat16, DEVICE, layout(torch.bfloat16))
    from kvmini.models.llama import LayerWeights, LlamaWeights, interleave_gate_up

    one = lambda: torch.ones(cfg.hidden_size, dtype=torch.bfloat16, device=DEVICE)  # noqa: E731
    layers = []
    for i in range(cfg.num_layers):
        m = lambda n: get(f"l{i}.{n}")  # noqa: B023, E731
        layers.append(LayerWeights(one(), torch.cat((m("q"), m("k"), m("v"))), m("o"), one(), interleave_gate_up(m("gate"), m("up")).contiguous(), m("down")))
    return LlamaWeights(cfg, get("embed"), layers, one(), get("head"))


# ---- the passes ----------------------------------------------------------------------------------------------------
def _latencies(case: Dict[str, Any], seed: int) -> torch.Tensor:
    """Inter-token gaps in ms: log-normal around 12 ms, one in fifty of them a stall, one in a thousand missing."""
    shape = (case["metrics"], case["samples"])
    x = 12.0 * torch.exp(0.35 * _normal(seed, "gaps", shape))
    u = torch.rand(shape, generator=_generator(seed, "stalls"), device=DEVICE)
    x = torch.where(u < 0.02, x * 8, x)
    x = torch.where(u > 0.999, torch.full_like(x, float("nan")), x)
    return x.double() if case["double"] else x


@torch.no_grad()
def prepare(case: Dict[str, Any], seed: int) -> Dict[str, Any]:
    if case["design"] == "latencies":
        return {"samples": _latencies(case, seed)}
    from kvmini.engine.engine import EngineConfig, LLMEngine

    cfg = _config(case)
    tokens = _tokens(case, seed, cfg.vocab_size)
    longest, blocks = max(map(len, tokens)), sum(-(-len(t) // 16) for t in tokens)
    quantization = None if case["weights"] == "bf16" else case["weights"]
    eng = LLMEngine(EngineConfig(model=cfg.name, device=DEVICE, max_num_seqs=MAX_SEQS, max_batched_tokens=MAX_TOKENS, max_model_len=-(-longest // 64) * 64 + 64, num_blocks=blocks + 2,
                                 quantization=quantization, kv_cache_dtype="auto" if case["cache"] == "bf16" else case["cache"]), weights=_weights(cfg, _checkpoint(cfg, seed)))
    seqs = [eng.make_sequence(t) for t in tokens]
    new = [1 if case["kind"] == "decode" else len(t) for t in tokens]
    # the contexts: prompt steps of as many tokens as fit
    left = [(s, len(s.prompt_ids) - n) for s, n in zip(seqs, new)]
    while any(n for _s, n in left):
        budget, portions, rest = MAX_TOKENS, [], []
        for s, n in left:
            take = min(n, budget)
            budget -= take
            rest.append((s, n - take))
            if take:
                portions.append((s, take, []))
        batch = eng.scheduler.schedule_given(portions)
        eng.runner.execute(batch)
        eng.scheduler.note_computed(batch)
        left = rest
    eng.runner.capture_graphs([eng.runner.bucket_for(sum(new))])
    return {"engine": eng, "portions": [(s, n, _wanted(case, n)) for s, n in zip(seqs, new)], "pending": None, "hybrid": hasattr(eng.runner, "memory")}


@torch.no_grad()
def run(state: Dict[str, Any]) -> Any:
    if "samples" in state:
        from kvmini.ops.hist_quantile import batched_quantiles

        return batched_quantiles(state["samples"], LEVELS)
    eng = state["engine"]
    step = eng.runner.launch(eng.scheduler.schedule_given(state["portions"]))
    if state["pending"] is not None:
        eng.runner.collect(state["pending"])
    state["pending"] = step
    memory = [eng.runner.kv_cache] if not state["hybrid"] else \
        [t for layer in eng.runner.memory.runs for branch in layer for t in branch if t.shape[-1] != 2]  # (two bf16 hold one fp32 factor there)
    return {"logits": step.logits[: step.n_samples], "memory": memory}


def work(case: Dict[str, Any]) -> Dict[str, float]:
    if case["design"] == "latencies":
        n = case["metrics"] * case["samples"]
        return {"bytes": n * (8.0 if case["double"] else 4.0), "flops": 0.0}
    cfg, lengths = _config(case), _lengths(case)
    w, decode = cfg.hidden_size, case["kind"] == "decode"
    rows = len(lengths) if decode else sum(lengths)
    each = {"bf16": 2.0, "fp8": 1.0, "mxfp4": 0.53125}[case["weights"]]
    cell = 2.0 if case["cache"] == "bf16" else 1.0

    def seen(window: int = 0) -> float:
        """(Query, key) pairs."""
        reach = lambda n: min(n, window or n)  # noqa: E731
        return float(sum(reach(n + 1) for n in lengths) if decode else sum(reach(n) * (reach(n) + 1) / 2 + (n - reach(n)) * reach(n) for n in lengths))

    def cached(window: int = 0) -> float:
        return seen(window) if decode else float(rows)  # rows of the cache read, or written

    head = cfg.vocab_size * w
    mem = 2.0 * head + 2.0 * rows * w
    flops = 2.0 * head * sum(len(_wanted(case, 1 if decode else n)) for n in lengths)
    if case["design"] == "llama":
        params = sum(a * b for a, b in _llama_shapes(cfg).values())
        kv = cfg.num_kv_heads * cfg.head_dim
        mem += cfg.num_layers * (each * params + 2 * cell * cached() * kv)
        flops += cfg.num_layers * (2.0 * rows * params + 4.0 * seen() * cfg.num_heads * cfg.head_dim)
        return {"bytes": mem, "flops": flops}
    for la in cfg.layers:
        params = 0.0
        for b in la.branches:
            m, kind = b.mixer, type(b.mixer).__name__
            if kind == "AttentionSpec":
                row = m.kv_heads * (m.dim + (m.rot_dims if m.key_values else m.vdim))
                params += w * (m.heads * (m.dim + m.vdim) + m.kv_heads * (m.dim + (0 if m.key_values else m.vdim)) + m.gates)
                mem += 2.0 * cached(m.window) * row
                flops += 2.0 * seen(m.window) * m.heads * (m.dim + m.vdim)
            elif kind == "LatentSpec":
                row, both = m.kv_rank + m.rot_dim, m.heads * (m.dim + m.vdim)
                params += w * (m.heads * (m.dim + m.rot_dim + m.vdim) + (row if m.kv_from < 0 else 0) + m.gates) + m.kv_rank * both
                mem += 2.0 * cached(m.window) * row
                flops += 2.0 * seen(m.window) * (m.heads * (row + m.kv_rank) if decode else both + m.heads * m.rot_dim)
            elif kind == "DeltaSpec":
                inner, ranks = m.heads * m.vdim, (m.decay_rank or m.dim) + (m.gate_rank or m.dim)
                params += w * (m.channels + m.heads + inner + ranks) + (m.decay_rank or m.dim) * m.heads * m.dim + (m.gate_rank or m.dim) * inner
                mem += 8.0 * len(lengths) * m.heads * m.dim * m.vdim
                flops += 6.0 * rows * m.heads * m.dim * m.vdim
            elif kind == "RetentionSpec":
                params += w * m.heads * (2 * m.dim + 3 * m.vdim)
                mem += 8.0 * len(lengths) * m.heads * m.dim * m.vdim
                flops += 4.0 * rows * m.heads * m.dim * m.vdim
            else:
                params += w * (m.inner + m.channels + m.heads + m.inner)
                mem += 8.0 * len(lengths) * m.inner * m.dim
                flops += 4.0 * rows * m.inner * m.dim
        params += 3.0 * w * la.ff
        if cfg.wiring == "gated":
            params += w * w * (2 if la.feeds_forward else 1)
        mem += 2.0 * params
        flops += 2.0 * rows * params
        if la.moe is not None:
            e = la.moe
            touched = e.experts * (1.0 - (1.0 - e.top / e.experts) ** rows)
            n = 3 if e.gated else 2
            mem += 2.0 * w * (e.experts + n * (touched * e.ff + e.shared_ff))
            flops += 2.0 * rows * w * (e.experts + n * (e.top * e.ff + e.shared_ff))
    return {"bytes": mem, "flops": flops}


def tolerance(case: Dict[str, Any]) -> Any:
    if case["design"] == "latencies":
        return "exact"
    return {"rel": 0.03, "max": 0.5}


# ---- the same in 64 bits, from the weights as drawn ----------------------------------------------------------------
Spans = List[Tuple[int, int]]  # every sequence's rows


def _unit(x: torch.Tensor, eps: float) -> torch.Tensor:
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x: torch.Tensor) -> torch.Tensor:
    return x * torch.sigmoid(x)


def _turn(x: torch.Tensor, pos: torch.Tensor, base: float, dims: int, neighbours: bool = False) -> torch.Tensor:
    """x [T, heads, n]: pairs (i, i + dims / 2), or neighbours, of the first ``dims`` entries, by position * base^(-2i / dims)."""
    half = dims // 2
    a = pos[:, None, None].double() * base ** (-2.0 * torch.arange(half, device=x.device, dtype=torch.float64) / max(1, dims))
    c, s = a.cos(), a.sin()
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if neighbours else (x[..., :half], x[..., half:dims])
    p, q = u * c - v * s, v * c + u * s
    return torch.cat((torch.stack((p, q), -1).flatten(-2) if neighbours else torch.cat((p, q), -1), x[..., dims:]), -1)


def _softmax_attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, scale: float, spans: Spans, window: int = 0, keep: int = 0, sink: Optional[torch.Tensor] = None,
                       rel: Optional[torch.Tensor] = None) -> torch.Tensor:
    """q [T, H, d], k [T, G, d], v [T, G, dv] -> [T, H, dv]; ``rel`` [H, distances], the last one: and beyond."""
    nh, g = q.shape[1], k.shape[1]
    out = torch.empty((q.shape[0], nh, v.shape[2]), dtype=q.dtype, device=q.device)
    for a, b in spans:
        ks, vs = k[a:b].permute(1, 2, 0).contiguous(), v[a:b].transpose(0, 1).contiguous()
        size = max(16, min(1024, (1 << 28) // (nh * (b - a))))
        for i in range(a, b, size):
            j = min(b, i + size)
            n = j - a
            s = torch.matmul(q[i:j].transpose(0, 1).reshape(g, nh // g * (j - i), -1) * scale, ks[:, :, :n].contiguous()).view(nh, j - i, n)
            far = torch.arange(i - a, n, device=q.device)[:, None] - torch.arange(n, device=q.device)[None]
            if rel is not None:
                s += rel[:, far.clamp(0, rel.shape[1] - 1)]
            hidden = far < 0
            if window:
                hidden = hidden | ((far >= window) & (torch.arange(n, device=q.device) >= keep)[None])
            s.masked_fill_(hidden, -math.inf)
            top = s.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[:, None, None])
            s.sub_(top).exp_()
            total = s.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[:, None, None] - top)
            o = torch.matmul(s.view(g, nh // g * (j - i), n), vs[:, :n]).view(nh, j - i, -1) / total
            out[i:j] = o.transpose(0, 1)
    return out


def _walk(spans: Spans, inputs: List[torch.Tensor], state: Tuple[int, ...], out: Tuple[int, ...], step: Callable[..., Tuple[torch.Tensor, torch.Tensor]]) -> torch.Tensor:
    """Token by token, all sequences at once: (state, output) = step(state, *inputs of the token)."""
    dev, longest = inputs[0].device, max(b - a for a, b in spans)
    at = torch.stack([(a + torch.arange(longest, device=dev)).clamp(max=b - 1) for a, b in spans], 1)  # (a sequence that is over repeats its last token, unseen)
    s = torch.zeros((len(spans), *state), dtype=torch.float64, device=dev)
    y = torch.empty((inputs[0].shape[0], *out), dtype=torch.float64, device=dev)
    for t in range(longest):
        live = [i for i, (a, b) in enumerate(spans) if t < b - a]
        s, o = step(s, *(x[at[t]] for x in inputs))
        y[at[t][live]] = o[live]
    return y


def _convolve(x: torch.Tensor, taps: torch.Tensor, spans: Spans) -> torch.Tensor:
    """Causal, per channel; taps [channels, n], the last one is the current token's."""
    n, out = taps.shape[1], torch.empty_like(x)
    for a, b in spans:
        ext = torch.nn.functional.pad(x[a:b], (0, 0, n - 1, 0))
        out[a:b] = sum(ext[j : j + b - a] * taps[:, j] for j in range(n))
    return out


def _rounded(w: torch.Tensor, kind: str) -> torch.Tensor:
    """A matrix [out, in] as the quantised engine keeps it: e4m3 with a scale per row, or e2m1 with a power of two per 32."""
    x = w.float()
    if kind == "fp8":
        scale = x.abs().amax(1, keepdim=True).clamp_min(1e-12) / 448.0
        return (x / scale).to(torch.float8_e4m3fn).double() * scale.double()
    if kind == "mxfp4" and w.shape[1] % 256 == 0:
        b = x.view(w.shape[0], -1, 32)
        e = torch.exp2(torch.floor(torch.log2(b.abs().amax(-1, keepdim=True).clamp_min(2.0 ** -120))) - 2.0)
        y = (b / e).abs()
        grid = torch.where(y < 2, (y * 2).round() / 2, torch.where(y < 4, y.round(), (y / 2).round() * 2)).clamp(max=6.0)
        return (torch.sign(b) * grid * e).double().view(w.shape)
    return w.double()


class _Exact:
    """The models in 64 bits on all tokens of all sequences, ``pos`` each one's position."""

    def __init__(self, case: Dict[str, Any], seed: int):
        self.cfg, self.case = _config(case), case
        self.get = _checkpoint(self.cfg, seed)
        tokens = _tokens(case, seed, self.cfg.vocab_size)
        ends = np.cumsum([len(t) for t in tokens]).tolist()
        self.spans = list(zip([0] + ends[:-1], ends))
        self.ids = torch.tensor([t for s in tokens for t in s], device=DEVICE)
        self.pos = torch.cat([torch.arange(len(t), device=DEVICE) for t in tokens])
        new = [1 if case["kind"] == "decode" else len(t) for t in tokens]
        self.rows = torch.tensor([b - n + r for (_a, b), n in zip(self.spans, new) for r in _wanted(case, n)], device=DEVICE)

    def w(self, name: str) -> torch.Tensor:
        return self.get(name).double()

    def mul(self, x: torch.Tensor, name: str) -> torch.Tensor:
        return x @ self.w(name).T

    def norm(self, x: torch.Tensor, name: str) -> torch.Tensor:
        return _unit(x, self.cfg.rms_eps) * self.w(name)

    def llama(self) -> torch.Tensor:
        cfg, t = self.cfg, len(self.ids)
        x = self.w("embed")[self.ids]
        mul = lambda v, n: v @ _rounded(self.get(n), self.case["weights"]).T  # noqa: E731
        for i in range(cfg.num_layers):
            h = _unit(x, cfg.rms_eps)
            q, k, v = (mul(h, f"l{i}.{n}").view(t, -1, cfg.head_dim) for n in "qkv")
            q, k = (_turn(z, self.pos, cfg.rope_theta, cfg.head_dim) for z in (q, k))
            x = x + mul(_softmax_attention(q, k, v, cfg.head_dim ** -0.5, self.spans).reshape(t, -1), f"l{i}.o")
            h = _unit(x, cfg.rms_eps)
            x = x + mul(_silu(mul(h, f"l{i}.gate")) * mul(h, f"l{i}.up"), f"l{i}.down")
        return self.mul(_unit(x[self.rows], cfg.rms_eps), "head")

    def attention(self, h: torch.Tensor, m: Any, n: str) -> torch.Tensor:
        t = len(h)
        q, k = ((self.mul(h, f"{n}.{z}") + self.w(f"{n}.{z}.b")).view(t, -1, m.dim) for z in "qk")
        v = k if m.key_values else (self.mul(h, n + ".v") + self.w(n + ".v.b")).view(t, -1, m.vdim)
        sink = rel = None
        if m.key_values:  # (rotated ahead of the norm or behind it: the norm has no gains, so either is the same)
            q, k, sink = _unit(q, self.cfg.rms_eps), _unit(k, self.cfg.rms_eps), self.w(n + ".sink")
        else:
            q, k = _unit(q, self.cfg.rms_eps) * self.w(n + ".q.norm"), _unit(k, self.cfg.rms_eps) * self.w(n + ".k.norm")
        q, k = (_turn(z, self.pos, m.rot_base, m.rot_dims) for z in (q, k))
        if m.rel:
            table, half = self.w(n + ".rel"), m.rel_buckets / 2
            row = lambda d: d if d < half else min(m.rel_buckets - 1, int(half + math.floor(math.log(d / half) / math.log(m.rel_max / half) * (m.rel_buckets - half))))  # noqa: E731
            rel = table[[row(d) for d in range(max(m.rel_max, 1) + 1)]].T
        spans = self.spans
        if m.chunk:
            spans = [(i, min(b, i + m.chunk)) for a, b in self.spans for i in range(a, b, m.chunk)]
        o = _softmax_attention(q, k, v, m.scale, spans, m.window, m.keep, sink, rel)
        if m.gate == "head":
            o = o * torch.sigmoid(self.mul(h, n + ".g"))[:, :, None]
        o = o.reshape(t, -1)
        if m.gate == "element":
            o = o * torch.sigmoid(self.mul(h, n + ".g"))
        o = self.mul(o, n + ".o")
        return o + self.w(n + ".o.b") if m.out_bias else o

    def latent(self, h: torch.Tensor, m: Any, n: str, made: Dict[int, Any], layer: int) -> torch.Tensor:
        t = len(h)
        if m.kv_from < 0:
            z = self.mul(h, n + ".dkv")
            made[layer] = (self.norm(z[:, : m.kv_rank], n + ".dkv.norm"), _turn(z[:, None, m.kv_rank :], self.pos, m.rot_base, m.rot_dim, True))
        c, kr = made[layer if m.kv_from < 0 else m.kv_from]
        q = self.mul(h, n + ".q").view(t, m.heads, -1)
        q = torch.cat((q[..., : m.dim], _turn(q[..., m.dim :], self.pos, m.rot_base, m.rot_dim, True)), -1)
        k = torch.cat((self.mul(c, n + ".uk").view(t, m.heads, m.dim), kr.expand(t, m.heads, m.rot_dim)), -1)
        o = _softmax_attention(q, k, self.mul(c, n + ".uv").view(t, m.heads, m.vdim), m.scale, self.spans, m.window)
        g = torch.sigmoid(self.mul(h, n + ".g"))
        o = (o * g[:, :, None]).reshape(t, -1) if m.gate == "head" else o.reshape(t, -1) * g
        return self.mul(o, n + ".o")

    def delta(self, h: torch.Tensor, m: Any, n: str) -> torch.Tensor:
        t, rep = len(h), m.heads // m.kv_heads
        q, k, v = (_silu(_convolve(self.mul(h, f"{n}.{z}"), self.w(f"{n}.{z}.conv"), self.spans)).view(t, -1, m.vdim if z == "v" else m.dim) for z in "qkv")
        q, k = (z * torch.rsqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
        q, k = (z.repeat_interleave(rep, 1) for z in (q * m.dim ** -0.5, k))
        beta = torch.sigmoid(self.mul(h, n + ".b"))
        sp = torch.nn.functional.softplus(self.mul(self.mul(h, n + ".a1"), n + ".a2") + self.w(n + ".dt_bias")).view(t, m.heads, m.dim)
        decay = torch.exp(-torch.exp(self.w(n + ".A_log"))[:, None] * sp)

        def step(s: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, beta: torch.Tensor, decay: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
            s = s * decay[..., None]
            u = beta[..., None] * (v - (s * k[..., None]).sum(-2))
            s = s + k[..., None] * u[..., None, :]
            return s, (s * q[..., None]).sum(-2)

        o = _walk(self.spans, [q, k, v, beta, decay], (m.heads, m.dim, m.vdim), (m.heads, m.vdim), step)
        gate = torch.sigmoid(self.mul(self.mul(h, n + ".g1"), n + ".g2"))
        return self.mul((self.norm(o, n + ".norm")).reshape(t, -1) * gate, n + ".o")

    def retention(self, h: torch.Tensor, m: Any, n: str) -> torch.Tensor:
        t = len(h)
        q, k = (_turn(self.mul(h, f"{n}.{z}").view(t, m.heads, m.dim), self.pos, m.rot_base, m.rot_dims) for z in "qk")
        decay = torch.tensor(m.decay, dtype=torch.float64, device=DEVICE)[:, None, None]

        def step(s: torch.Tensor, q: torch.Tensor, k: torch.Tensor, v: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
            s = s * decay + k[..., None] * v[..., None, :]
            return s, (s * q[..., None]).sum(-2)

        o = _walk(self.spans, [q, k * m.dim ** -0.5, self.mul(h, n + ".v").view(t, m.heads, m.vdim)], (m.heads, m.dim, m.vdim), (m.heads, m.vdim), step)
        return self.mul(_unit(o, self.cfg.rms_eps).reshape(t, -1) * _silu(self.mul(h, n + ".g")), n + ".o")

    def state_space(self, h: torch.Tensor, m: Any, n: str) -> torch.Tensor:
        t, rep = len(h), m.heads // m.groups
        z, xbc, dt = self.mul(h, n + ".in").split((m.inner, m.channels, m.heads), -1)
        xbc = _silu(_convolve(xbc, self.w(n + ".conv"), self.spans) + self.w(n + ".conv.b"))
        x, b, c = xbc.split((m.inner, m.groups * m.dim, m.groups * m.dim), -1)
        x, b, c = x.reshape(t, m.heads, m.vdim), b.reshape(t, m.groups, m.dim), c.reshape(t, m.groups, m.dim)
        dt = torch.nn.functional.softplus(dt + self.w(n + ".dt_bias"))
        decay = torch.exp(-torch.exp(self.w(n + ".A_log")) * dt)

        def step(s: torch.Tensor, x: torch.Tensor, b: torch.Tensor, c: torch.Tensor, dt: torch.Tensor, decay: torch.Tensor) -> Tuple[torch.Tensor, torch.Tensor]:
            b, c = (y.repeat_interleave(rep, 1) for y in (b, c))
            s = s * decay[..., None, None] + (dt[..., None] * b)[..., None] * x[..., None, :]
            return s, (s * c[..., None]).sum(-2)

        y = _walk(self.spans, [x, b, c, dt, decay], (m.heads, m.dim, m.vdim), (m.heads, m.vdim), step) + self.w(n + ".D")[:, None] * x
        y = y.reshape(t, -1) * _silu(z)
        y = _unit(y.view(t, m.norm_groups, -1), self.cfg.rms_eps).reshape(t, -1) * self.w(n + ".norm")
        return self.mul(y, n + ".o")

    def mixer(self, h: torch.Tensor, i: int, made: Dict[int, Any]) -> torch.Tensor:
        y = 0.0
        for b in self.cfg.layers[i].branches:
            m, n, kind = b.mixer, f"l{i}.{b.tensors}", type(b.mixer).__name__
            if kind == "LatentSpec":
                o = self.latent(h, m, n, made, i)
            else:
                o = {"AttentionSpec": self.attention, "DeltaSpec": self.delta, "RetentionSpec": self.retention, "StateSpaceSpec": self.state_space}[kind](h, m, n)
            y = y + b.scale * o
        return y

    def gated(self, h: torch.Tensor, n: str, act: Any, limit: float = math.inf) -> torch.Tensor:
        if act == "relu2":
            return self.mul(torch.relu(self.mul(h, n + "up")) ** 2, n + "down")
        g, u = self.mul(h, n + "gate"), self.mul(h, n + "up")
        if act == "clamped":
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            return self.mul(g * torch.sigmoid(1.702 * g) * (u + 1), n + "down")
        return self.mul((_silu(g) if act == "silu" else torch.nn.functional.gelu(g, approximate="tanh")) * u, n + "down")

    def feed_forward(self, h: torch.Tensor, i: int) -> torch.Tensor:
        la, n = self.cfg.layers[i], f"l{i}.mlp."
        e = la.moe
        if e is None:
            return self.gated(h, n, la.act)
        z = self.mul(h, n + "router") + (self.w(n + "router.b") if e.bias else 0.0)
        scores = torch.sigmoid(z) if e.scores == "sigmoid" else z.softmax(-1)
        idx = (scores + (self.w(n + "correction") if e.correction else 0.0)).topk(e.top, dim=-1).indices
        share = z.gather(-1, idx).softmax(-1) if e.scores == "chosen" else scores.gather(-1, idx)
        y = torch.zeros_like(h)
        for j in range(e.experts):
            at, place = (idx == j).nonzero(as_tuple=True)
            if len(at):
                y[at] += e.scale * share[at, place][:, None] * self.gated(h[at], f"{n}e{j}.", e.act, e.limit)
        if e.shared_ff:
            s = self.gated(h, n + "shared.", e.act)
            y += s * torch.sigmoid(self.mul(h, n + "shared.sg")) if e.shared_gate else s
        return y

    def hybrid(self) -> torch.Tensor:
        cfg, eps, made = self.cfg, self.cfg.rms_eps, {}
        x = self.w("embed")[self.ids] * cfg.embed_scale
        width = x.shape[1]
        if cfg.sine_positions:
            a = self.pos[:, None].double() * 10000.0 ** (-2.0 * torch.arange(width // 2, device=DEVICE, dtype=torch.float64) / width)
            x = x + torch.stack((a.sin(), a.cos()), -1).flatten(-2)
        if cfg.wiring == "hyper":
            x = x[None].repeat(cfg.streams, 1, 1)
        for i, la in enumerate(cfg.layers):
            n = f"l{i}."
            mix, ff = (lambda h: self.mixer(h, i, made)), (lambda h: self.feed_forward(h, i))  # noqa: B023
            subs = [("1", mix)] + ([("2", ff)] if la.feeds_forward else [])
            if cfg.wiring == "parallel":
                x = x + sum(f(self.norm(x, f"{n}norm{s}")) for s, f in subs)
                continue
            for s, f in subs:
                if cfg.wiring == "hyper":
                    p = f"{n}hc{s}."
                    y = f(self.norm((self.w(p + "in")[:, None, None] * x).sum(0), f"{n}norm{s}"))
                    x = (self.w(p + "mix").T @ x.flatten(1)).view(x.shape) + self.w(p + "out")[:, None, None] * y
                elif cfg.wiring == "sandwich":
                    x = x + self.norm(f(self.norm(x, f"{n}norm{s}")), f"{n}norm{s}b")
                else:
                    y = f(x) * torch.sigmoid(self.mul(x, f"{n}rg{s}") + self.w(f"{n}rg{s}.b"))
                    x = x + cfg.residual_mult * self.norm(y, f"{n}norm{s}")
        x = (x.sum(0) if cfg.wiring == "hyper" else x)[self.rows]
        z = self.mul(self.norm(x, "final.norm"), "embed" if cfg.tied_head else "head") * cfg.logit_scale
        return cfg.logit_softcap * torch.tanh(z / cfg.logit_softcap) if cfg.logit_softcap else z


@torch.no_grad()
def exact(case: Dict[str, Any], seed: int) -> Any:
    if case["design"] == "latencies":
        out = np.full((case["metrics"], len(LEVELS)), np.nan)
        for i, row in enumerate(_latencies(case, seed).double()):
            v = row[~row.isnan()].sort().values
            for j, p in enumerate(LEVELS):
                at = p * (v.numel() - 1)
                lo, hi = v[math.floor(at)].item(), v[math.ceil(at)].item()
                out[i, j] = lo if lo == hi else lo + (at - math.floor(at)) * (hi - lo)
        return out
    e = _Exact(case, seed)
    # (the sequences' memory is laid out as the engine likes it)
    return {"logits": e.llama() if case["design"] == "llama" else e.hybrid(), "memory": None}
