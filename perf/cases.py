"""The workloads this framework is timed on.

A case is one unit of a user's work through the package's public entry points:

* "decode": one decode step of a stack of MoE layers, each layer one
  `ProgressiveReader` call on its own routed batch. The layers share one
  workspace and are captured in one HIP graph, as a serving engine runs them
  (`graph`); a larger batch, and a mode that enqueues torch operations of its
  own, is called eagerly.
* "sketch": the resident sketch of one layer's gate/up rows (`build_sketch`),
  which a program that loads a model makes once for each of its layers.

Shapes are those of the benchmark and the tests: OLMoE-1B-7B, Qwen3-30B-A3B, a
256-expert layer, Gemma 4 and Qwen3-235B-A22B. Weights are N(0, 0.02^2) in
BF16; hidden states N(0, 1) with 1 % of the dimensions scaled by 20; experts
come from a softmax router, or from a Zipf popularity law by Gumbel top-k; the
recovery map projects the down columns onto a random orthonormal basis.
"""

from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(
    0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "calibration-free-moe_amd")
)

from calibration_free_moe.reader.budget import compile_budget  # noqa: E402
from calibration_free_moe.reader.progressive import (  # noqa: E402
    ProgressiveReader,
    channel_major_down,
)
from calibration_free_moe.reader.sketch import block_hadamard_signs, build_sketch  # noqa: E402

# hidden, width, experts, top-k, activation
SHAPES = {
    "olmoe": (2048, 1024, 64, 8, "silu"),
    "qwen3": (2048, 768, 128, 8, "silu"),
    "fine256": (2048, 512, 256, 8, "silu"),
    "gemma4": (2816, 704, 128, 8, "gelu_tanh"),
    "qwen235": (4096, 1536, 128, 8, "silu"),
}

DECODE = {
    "kind": "decode", "layers": 4, "rank": 32, "retention": 0.123, "keep": 0.625,
    "score": "point", "zipf": 0.0, "threshold": False, "ids64": True, "weights16": False,
    "padded": 0, "graph": True,
}


def _decode(name: str, shape: str, tokens: int, **options: object) -> dict:
    return {"name": name, **DECODE, "shape": shape, "tokens": tokens, **options}


def listed() -> list[dict]:
    return [
        # the smallest call there is: one token through one layer, called
        # directly (a first token, a debugger, an engine without graphs)
        _decode("qwen3-t1-call", "qwen3", 1, layers=1, graph=False),
        # single-stream decoding, the latency-bound headline: one token, a
        # stack of layers in a graph
        _decode("qwen3-t1", "qwen3", 1, layers=8),
        # a handful of streams on the fine-grained layer; 5 is no multiple of
        # anything, and the batch is below the grouped schedule
        _decode("fine256-t5", "fine256", 5, layers=6),
        # a small batch with the reader's default (recovery-aware) score,
        # padded by the engine to its capture size
        _decode("qwen3-t13of16-aware", "qwen3", 16, padded=3, score="recovery-aware"),
        # Gemma 4: hidden size 2816, GELU, the default score, BF16 router
        # weights and int32 ids as vLLM's fused router gives them
        _decode("gemma4-t24-aware", "gemma4", 24, score="recovery-aware", weights16=True,
                ids64=False),
        # calibrated-threshold selection (its read statistics follow the
        # selection), a rank-16 recovery map, an odd batch
        _decode("qwen3-t31-threshold-r16", "qwen3", 31, layers=2, rank=16, threshold=True,
                graph=False),
        # the widest layer supported in earnest: Qwen3-235B at a busy batch
        _decode("qwen235-t48", "qwen235", 48, layers=1),
        # the benchmark's headline: OLMoE at batch 64
        _decode("olmoe-t64", "olmoe", 64),
        # a full decode batch
        _decode("qwen3-t128", "qwen3", 128),
        # skewed routing at a large batch, a generous budget and the full
        # screen, a rank-64 map
        _decode("qwen3-t256-zipf", "qwen3", 256, layers=2, retention=0.25, keep=1.0, rank=64,
                zipf=1.2),
        # the largest batch a call takes (8192 routed pairs), ragged
        _decode("qwen3-t1000", "qwen3", 1000, layers=1, graph=False),
        # model loading: the sketch of one layer
        {"name": "sketch-qwen3", "kind": "sketch", "hidden": 2048, "width": 768, "experts": 128},
    ]


def draw(rng) -> dict:
    """One more case of the ranges the listed ones stand for."""
    if rng.random() < 0.12:
        hidden = 128 * rng.randint(8, 32)
        width = 16 * rng.randint(16, 96)
        experts = max(4, min(128, int(0.2e9 / (2 * width * hidden))))
        return {"kind": "sketch", "hidden": hidden, "width": width,
                "experts": rng.randint(max(2, experts // 3), experts)}
    shape = rng.choice(sorted(SHAPES))
    limit = 160 if shape == "qwen235" else 700
    tokens = min(limit, max(1, round(math.exp(rng.uniform(0.0, math.log(limit + 1))))))
    graph = tokens <= 256 and (tokens > 1 or rng.random() < 0.7)
    threshold = rng.random() < 0.12
    case = {
        **DECODE, "shape": shape, "tokens": tokens,
        "layers": 1 if shape == "qwen235" or tokens > 256 or not graph else 2,
        "rank": rng.choice([32, 32, 32, 16, 64]),
        "retention": rng.choice([0.06, 0.123, 0.123, 0.125, 0.2, 0.25]),
        "keep": rng.choice([0.625, 0.625, 1.0]),
        "score": "point" if threshold else rng.choice(["point", "recovery-aware"]),
        "zipf": rng.choice([0.0, 0.0, 1.2]),
        "threshold": threshold,
        "ids64": rng.random() < 0.5,
        "weights16": rng.random() < 0.3,
        "padded": rng.randint(1, max(1, tokens // 8)) if tokens >= 4 and rng.random() < 0.3 else 0,
        "graph": graph and not threshold,
    }
    return case


# ---------------------------------------------------------------------------
# inputs


def _device() -> torch.device:
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed: int, stream: int) -> torch.Generator:
    return torch.Generator(device=_device()).manual_seed(seed * 1009 + stream)


def _normal(shape: tuple[int, ...], std: float, g: torch.Generator) -> torch.Tensor:
    return torch.empty(shape, dtype=torch.bfloat16, device=_device()).normal_(0.0, std, generator=g)


def _weights(case: dict, seed: int, layer: int) -> dict[str, torch.Tensor]:
    """One layer's gate/up rows, down columns, recovery map and router."""
    hidden, width, experts, _, _ = SHAPES[case["shape"]]
    g = _generator(seed, 2 * layer)
    gate_up = _normal((experts, 2 * width, hidden), 0.02, g)
    down = _normal((experts, hidden, width), 0.02, g)
    router = _normal((experts, hidden), 0.02, g)
    basis = torch.randn(hidden, case["rank"], generator=g, device=_device())
    decoder = torch.linalg.qr(basis).Q.bfloat16().contiguous()
    projection = decoder.T.contiguous()
    encoder = torch.stack([projection @ down[e] for e in range(experts)])
    return {"gate_up": gate_up, "down": down, "router": router, "decoder": decoder,
            "encoder": encoder}


def _batch(case: dict, router: torch.Tensor, tokens: int, g: torch.Generator) -> dict:
    """A routed batch of one layer."""
    hidden, _, experts, top_k, _ = SHAPES[case["shape"]]
    device = _device()
    x = torch.randn(tokens, hidden, generator=g, device=device)
    dims = torch.randperm(hidden, generator=g, device=device)[: max(1, round(0.01 * hidden))]
    x[:, dims] *= 20.0
    x = x.bfloat16()
    if case["zipf"]:
        rank = torch.arange(1, experts + 1, dtype=torch.float64, device=device)
        log_p = -case["zipf"] * torch.log(rank)
        log_p = log_p[torch.randperm(experts, generator=g, device=device)]
        uniform = torch.rand(tokens, experts, generator=g, device=device, dtype=torch.float64)
        logits = log_p - torch.log(-torch.log(uniform))
        top = logits.topk(top_k, dim=-1)
        weights, ids = torch.softmax(top.values, dim=-1), top.indices
    else:
        logits = (x.float() @ router.float().T).bfloat16().float()
        weights, ids = torch.softmax(logits, -1).topk(top_k, -1)
        weights = weights / weights.sum(-1, keepdim=True)
    weights = weights.to(torch.bfloat16 if case["weights16"] else torch.float32).contiguous()
    ids = ids.to(torch.int64 if case["ids64"] else torch.int32).contiguous()
    padding = None
    if case["padded"]:
        padding = torch.arange(tokens, device=device) >= tokens - case["padded"]
    return {"x": x, "ids": ids, "weights": weights, "padding": padding}


def _plan(case: dict):
    hidden, width, _, top_k, _ = SHAPES[case["shape"]]
    return compile_budget(hidden_size=hidden, expert_width=width, top_k=top_k,
                          retention=case["retention"], screen_keep=case["keep"])


CALIBRATION_TOKENS = 16  # rows a selection threshold is calibrated on


def _calibration(case: dict, router: torch.Tensor, seed: int, layer: int) -> dict:
    return _batch({**case, "padded": 0}, router, CALIBRATION_TOKENS, _generator(seed, 90 + layer))


def prepare(case: dict, seed: int) -> dict:
    device = _device()
    if case["kind"] == "sketch":
        rows = _normal((case["experts"], 2 * case["width"], case["hidden"]), 0.02,
                       _generator(seed, 0))
        return {"kind": "sketch", "rows": rows,
                "signs": block_hadamard_signs(case["hidden"], device)}
    hidden, width, experts, _, activation = SHAPES[case["shape"]]
    plan, tokens = _plan(case), case["tokens"]
    calls, workspace = [], None
    for layer in range(case["layers"]):
        w = _weights(case, seed, layer)
        signs = block_hadamard_signs(hidden, device)
        sketch = build_sketch(w["gate_up"], signs, device_kernel=True)
        down = channel_major_down(w["down"])
        common = dict(sketch=sketch, activation=activation, selection_score=case["score"])
        threshold = None
        if case["threshold"]:
            probe = ProgressiveReader(w["gate_up"], down, w["encoder"], w["decoder"], plan,
                                      CALIBRATION_TOKENS, **common)
            b = _calibration(case, w["router"], seed, layer)
            probe(b["x"], b["ids"], b["weights"])
            cutoffs = probe.scores[0].topk(plan.final_count, dim=-1).values[:, -1]
            threshold = cutoffs.median().item()
        reader = ProgressiveReader(w["gate_up"], down, w["encoder"], w["decoder"], plan, tokens,
                                   workspace=workspace, selection_threshold=threshold, **common)
        workspace = reader.workspace
        b = _batch(case, w["router"], tokens, _generator(seed, 2 * layer + 1))
        calls.append((reader, b["x"], b["ids"], b["weights"], b["padding"],
                      torch.empty_like(b["x"])))
    state = {"kind": "decode", "calls": calls, "graph": None}
    if case["graph"]:
        # the kernels' code is on the device before the capture; the capture's
        # warm-up leaves no read statistics behind
        _step(calls)
        for reader, *_ in calls:
            reader.read_work.zero_()
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            _step(calls)
    return state


def _step(calls: list[tuple]) -> None:
    for reader, x, ids, weights, padding, out in calls:
        reader(x, ids, weights, padding, out)


def run(state: dict) -> dict:
    if state["kind"] == "sketch":
        codes, statistics = build_sketch(state["rows"], state["signs"], device_kernel=True)
        return {"codes": codes, "statistics": statistics}
    if state["graph"] is not None:
        state["graph"].replay()
    else:
        _step(state["calls"])
    return {"out": [call[5] for call in state["calls"]],
            "reads": [call[0].read_work for call in state["calls"]]}


# ---------------------------------------------------------------------------
# work and tolerances


def _touch_probabilities(case: dict) -> list[float]:
    """Each expert's probability of being among a token's top-k."""
    _, _, experts, top_k, _ = SHAPES[case["shape"]]
    if not case["zipf"]:
        return [top_k / experts] * experts
    p = [(r + 1) ** -case["zipf"] for r in range(experts)]
    # top-k without replacement: 1 - (1 - p)^m with the m that gives k experts a token
    total = sum(p)
    low, high = 1.0, 1e6
    for _ in range(60):
        m = math.sqrt(low * high)
        low, high = (m, high) if sum(1 - (1 - v / total) ** m for v in p) < top_k else (low, m)
    return [1 - (1 - v / total) ** low for v in p]


def work(case: dict) -> dict:
    """Bytes and operations one pass needs: every touched expert's sketch (the
    kept coordinates' codes and FP16 scales), norms, the union of its kept
    channels' rows and of its skipped channels' encoder rows (expected values),
    the decoder, and the batch in and out."""
    if case["kind"] == "sketch":
        values = case["experts"] * 2 * case["width"] * case["hidden"]
        # rows in; five trits to a byte and two FP16 statistics per block out;
        # seven butterflies and about nine operations per value
        return {"bytes": 2 * values + values / 5 + 4 * values / 128, "flops": 16 * values}
    hidden, width, _, top_k, _ = SHAPES[case["shape"]]
    plan, rank = _plan(case), case["rank"]
    tokens = case["tokens"] - case["padded"]
    keep, share = plan.screen_coordinates / 128, plan.final_count / plan.candidate_count
    planes = 1 if case["score"] == "point" else 2
    total = 0.0
    for q in _touch_probabilities(case):
        touched = 1 - (1 - q) ** tokens
        codes = hidden * (1 - (1 - q * keep) ** tokens) * 2 * math.ceil(width / 5)
        scales = touched * (hidden // 128) * 4 * width * planes
        selection = touched * 4 * width * (1 if planes == 1 else 3)
        kept = width * (1 - (1 - q * share) ** tokens)
        skipped = width * (1 - (1 - q * (1 - share)) ** tokens)
        total += codes + scales + selection + 6 * hidden * kept + 2 * rank * skipped
    total += 2 * hidden * rank + hidden + tokens * (4 * hidden + 8 * top_k)
    flops = tokens * (
        2 * 2 * plan.candidate_count * hidden * keep  # screen
        + 2 * 3 * plan.final_count * hidden  # kept rows
        + 2 * rank * (plan.candidate_count - plan.final_count + hidden)  # recovery
    )
    return {"bytes": case["layers"] * total, "flops": case["layers"] * flops}


def tolerance(case: dict) -> dict:
    # sketch: FP16 statistics (2^-11); a trit may differ where a magnitude lies
    # within an FP32 rounding of its threshold
    if case["kind"] == "sketch":
        return {"rel": 2e-4, "max": 2e-3, "differ": 1e-5}
    # BF16 outputs of sums over BF16 activations and slot values
    return {"rel": 1e-2, "max": 0.2}


# ---------------------------------------------------------------------------
# the same in 64 bits


def _hadamard(device: torch.device) -> torch.Tensor:
    h = torch.ones(1, 1, dtype=torch.float64, device=device)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / math.sqrt(128.0)


def _rotated(x: torch.Tensor, signs: torch.Tensor, hadamard: torch.Tensor) -> torch.Tensor:
    blocks = x.shape[-1] // 128
    return (x * signs).reshape(*x.shape[:-1], blocks, 128) @ hadamard


def _ternary(v: torch.Tensor) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Trits, scale and mean squared residual of 128-coordinate blocks."""
    magnitude = v.abs()
    above = magnitude > 0.7 * magnitude.mean(-1, keepdim=True)
    scale = (magnitude * above).sum(-1) / above.sum(-1).clamp_min(1)
    trits = torch.where(above, v.sign(), torch.zeros_like(v))
    residual = (v - trits * scale[..., None]).square().mean(-1)
    return trits, scale, residual


def _phi(gate: torch.Tensor, activation: str) -> torch.Tensor:
    if activation == "gelu_tanh":
        return torch.nn.functional.gelu(gate, approximate="tanh")
    return torch.nn.functional.silu(gate)


def _round16(v: torch.Tensor) -> torch.Tensor:
    return v.to(torch.bfloat16).double()


# five-point Gauss-Hermite rule of the standard normal
NODES = (-2.8569700138728056, -1.355626179974266, 0.0, 1.355626179974266, 2.8569700138728056)
MASSES = (0.011257411327720693, 0.2220759220056126, 0.5333333333333333, 0.2220759220056126,
          0.011257411327720693)


def _screened(case: dict, w: dict, b: dict, signs: torch.Tensor, hadamard: torch.Tensor):
    """Sketch projections [T, K, I] (gate, up) and the channel scores."""
    hidden, width, _, top_k, activation = SHAPES[case["shape"]]
    keep = _plan(case).screen_coordinates
    x, ids = b["x"].double(), b["ids"].long()
    tokens = x.shape[0]
    v = _rotated(x, signs, hadamard)  # [T, B, 128]
    kept = v.abs().argsort(dim=-1, descending=True, stable=True)[..., :keep]
    masked = torch.zeros_like(v).scatter(-1, kept, v.gather(-1, kept))
    energy = masked.square().sum(-1)  # [T, B]
    shape = (tokens, top_k, width)
    gate, up, scores = (torch.zeros(shape, dtype=torch.float64, device=x.device) for _ in range(3))
    live = torch.ones(tokens, dtype=torch.bool, device=x.device)
    if b["padding"] is not None:
        live = ~b["padding"]
    decoder = w["decoder"].double()
    gram = decoder.T @ decoder
    for e in torch.unique(ids[live]).tolist():
        t, k = torch.nonzero((ids == e) & live[:, None], as_tuple=True)
        trits, scale, residual = _ternary(_rotated(w["gate_up"][e].double(), signs, hadamard))
        scale, residual = scale.half().double(), residual.half().double()
        rows = (trits * scale[..., None]).reshape(2 * width, hidden)
        g, u = (masked[t].reshape(-1, hidden) @ rows.T).chunk(2, dim=-1)
        gate[t, k], up[t, k] = g, u
        down = w["down"][e].double()  # [H, I]
        norm = down.square().sum(0).sqrt()
        g, u = _round16(g), _round16(u)
        if case["score"] == "point":
            risk = (norm * _phi(g, activation) * u).square()
        else:
            sg, su = (energy[t] @ residual.T).chunk(2, dim=-1)
            sg = sg.sqrt()
            coder = w["encoder"][e].double()  # [R, I]
            alpha = (coder * (decoder.T @ down)).sum(0) / norm
            beta = ((coder * (gram @ coder)).sum(0) - alpha.square()).clamp_min(0).sqrt()
            first = energy_ = 0.0
            for node, mass in zip(NODES, MASSES):
                a = _phi(g + node * sg, activation)
                energy_ = energy_ + mass * a.square() * (u.square() + su)
                first = first + mass * a * u
            paid = _round16(_phi(g, activation) * u)
            risk = (norm.square() * (energy_ - first.square()).clamp_min(0)
                    + (norm * first - alpha * paid).square() + (beta * paid).square())
        scores[t, k] = risk * b["weights"].double()[t, k, None].square()
    return gate, up, scores, live


def _top(scores: torch.Tensor, count: int) -> torch.Tensor:
    """Mask of each row's `count` largest scores, ties to the lowest index."""
    order = scores.argsort(dim=-1, descending=True, stable=True)[:, :count]
    return torch.zeros_like(scores, dtype=torch.bool).scatter(1, order, True)


def _layer_exact(case: dict, seed: int, layer: int) -> torch.Tensor:
    hidden, width, _, top_k, activation = SHAPES[case["shape"]]
    device = _device()
    w = _weights(case, seed, layer)
    b = _batch(case, w["router"], case["tokens"], _generator(seed, 2 * layer + 1))
    bits = torch.randint(0, 2, (hidden,), generator=torch.Generator().manual_seed(0))
    signs, hadamard = (2 * bits - 1).to(device).double(), _hadamard(device)
    final = _plan(case).final_count
    gate, up, scores, live = _screened(case, w, b, signs, hadamard)
    tokens = gate.shape[0]
    flat = scores.reshape(tokens, -1)
    # candidates are numbered by expert id, then channel
    order = b["ids"].long().argsort(dim=-1, stable=True)
    by_expert = scores.gather(1, order[..., None].expand(-1, -1, width)).reshape(tokens, -1)
    if case["threshold"]:
        calibration = _calibration(case, w["router"], seed, layer)
        cutoffs = _screened(case, w, calibration, signs, hadamard)[2].reshape(CALIBRATION_TOKENS, -1)
        threshold = cutoffs.topk(final, dim=-1).values[:, -1].median()
        kept = _top(by_expert, final) & (by_expert >= threshold)
    else:
        kept = _top(by_expert, final)
    mask = torch.zeros_like(flat, dtype=torch.bool).reshape(scores.shape)
    mask.scatter_(1, order[..., None].expand(-1, -1, width), kept.reshape(scores.shape))
    out = torch.zeros(tokens, hidden, dtype=torch.float64, device=device)
    latent = torch.zeros(tokens, case["rank"], dtype=torch.float64, device=device)
    x, ids, weights = b["x"].double(), b["ids"].long(), b["weights"].double()
    for e in torch.unique(ids[live]).tolist():
        t, k = torch.nonzero((ids == e) & live[:, None], as_tuple=True)
        g, u = (x[t] @ w["gate_up"][e].double().T).chunk(2, dim=-1)
        chosen = mask[t, k]
        exact_ = torch.where(chosen, _phi(g, activation) * u, 0.0)
        sketched = torch.where(chosen, 0.0, _phi(gate[t, k], activation) * up[t, k])
        scale = weights[t, k, None]
        out.index_add_(0, t, scale * (exact_ @ w["down"][e].double().T))
        latent.index_add_(0, t, scale * (sketched @ w["encoder"][e].double().T))
    return out + latent @ w["decoder"].double().T


def exact(case: dict, seed: int):
    if case["kind"] == "sketch":
        state_rows = _normal((case["experts"], 2 * case["width"], case["hidden"]), 0.02,
                             _generator(seed, 0))
        device = _device()
        bits = torch.randint(0, 2, (case["hidden"],), generator=torch.Generator().manual_seed(0))
        signs, hadamard = (2 * bits - 1).to(device).double(), _hadamard(device)
        found = []
        for e in range(case["experts"]):
            _, scale, residual = _ternary(_rotated(state_rows[e].double(), signs, hadamard))
            found.append(torch.stack([scale, residual], dim=-1))
        return {"codes": None, "statistics": torch.stack(found)}
    return {"out": [_layer_exact(case, seed, layer) for layer in range(case["layers"])],
            "reads": [None] * case["layers"]}
