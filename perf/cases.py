"""The workloads this framework's speed is judged by, each one pass through its public entry points.

A case names the entry point (``path``) and its sizes.  The paths:

* ``decode``     -- one token's MoE MLP from its router logits (``moe_mlp_from_router_logits``): the step a chat
  repeats for every layer and every generated token.
* ``layer``      -- the MoE layer of some tokens whose routes are known (``prefill_moe_from_routes``): batched decode,
  prompt chunks, whole prompts.
* ``logits``     -- the same from the router logits on (``prefill_moe_from_router_logits``): routing included.
* ``fp8``        -- the routed experts with FP8 activations (``routed_experts(activations="float8_e4m3fn")``).
* ``share``      -- one GPU's part of an expert-parallel layer (``routed_experts_share``): its FP32 partial sum.
* ``projection`` -- the decode projection by itself (``fp8_routed_projection``): one row per route slot.
* ``panels``     -- a layer's routed half put together from the kernel interface: route grouping, row gather, M32
  panels, the panel matmuls, SwiGLU and the restore.

Expert tables are e4m3fn bytes with FP32 128x128 block scales quantised from N(0, 0.02), hidden rows and router logits
N(0, 1) (plus a Zipf popularity where ``zipf`` is not 0), the correction bias N(0, 0.05) (0 beside a Zipf popularity,
whose scores it would outweigh), shared tables N(0, 0.02).
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "glm-tpu_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from glm_moe.contracts import single_gpu_contract  # noqa: E402
from glm_moe.kernels.fp8_grouped_matmul.kernel import fp8_routed_projection  # noqa: E402
from glm_moe.kernels.fp8_grouped_matmul.panel_kernel import prefill_panel_fp8_matmul  # noqa: E402
from glm_moe.kernels.fp8_grouped_matmul.panels import build_expert_panels  # noqa: E402
from glm_moe.layers.moe.routed_experts import (  # noqa: E402
    gather_prefill_route_rows,
    group_prefill_routes,
    moe_mlp_from_router_logits,
    prefill_moe_from_router_logits,
    prefill_moe_from_routes,
    restore_prefill_route_rows,
    routed_experts,
    routed_experts_share,
    swiglu_bf16,
)

BLOCK = 128
ROUTED_SCALE = 2.5


def _case(name, path, tokens, *, experts=256, hidden=6144, inter=2048, top_k=8, zipf=0.0, shares=1, rank=0, tables=2,
          dtype="bfloat16"):
    case = dict(path=path, tokens=tokens, experts=experts, hidden=hidden, inter=inter, top_k=top_k, zipf=zipf)
    if path == "share":
        case.update(shares=shares, rank=rank)
    if path == "projection":
        case.update(tables=tables, dtype=dtype)
    if path == "panels":
        case.update(dtype=dtype)
    return case if name is None else dict(case, name=name)


def listed():
    return [
        # the smallest layer (the test fixture's scale): launches and host time are all there is
        _case("toy_t4", "layer", 4, experts=8, hidden=256, inter=256, top_k=2),
        # one chat generating: a token through a GLM-5-shape layer, router logits to layer output
        _case("decode_t1", "decode", 1),
        # four chats generating together
        _case("decode_t4", "layer", 4),
        # the decode projection that a program with its own layer body calls: gate and up of one token's 8 routes
        _case("projection_s8", "projection", 8, dtype="float32"),
        # about 64 chats generating together, one of them just gone
        _case("batch_t61", "layer", 61),
        # the reference engine's prefill block of 128 rows, from the logits
        _case("prefill_t128", "logits", 128),
        # the ragged last chunk of a prompt
        _case("prefill_t777", "layer", 777),
        # a prompt of 2048 tokens, evenly popular experts
        _case("prefill_t2048", "layer", 2048),
        # a long prompt from the logits on, a few experts taking most tokens
        _case("prefill_t8192_zipf", "logits", 8192, zipf=1.2),
        # a prompt in the FP8 activation mode
        _case("prefill_t2048_fp8", "fp8", 2048),
        # one of eight expert-parallel GPUs' part of a prompt
        _case("share8_t2048", "share", 2048, shares=8, rank=3),
        # a layer body put together from the kernel interface by the caller, an odd chunk
        _case("panels_t500", "panels", 500),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    path = rng.choice(("decode", "layer", "layer", "layer", "logits", "logits", "fp8", "share", "projection", "panels"))
    size = {}
    if path == "decode" or rng.random() < 0.4:  # another model's layer: smaller experts, fewer of them
        step = 512 if path == "projection" else 256
        size = dict(experts=rng.choice((16, 32, 64, 96, 128, 256)), hidden=step * rng.randint(2, 6144 // step),
                    inter=step * rng.randint(1, 2048 // step), top_k=rng.randint(2, 8))
    top_k = size.get("top_k", 8)
    experts = size.get("experts", 256)
    if path == "decode":
        return _case(None, path, 1, **size)
    if path == "projection":
        return _case(None, path, _log_int(rng, 1, 64), tables=rng.randint(1, 2),
                     dtype=rng.choice(("float32", "bfloat16")), **size)
    zipf = rng.choice((0.0, 0.0, round(rng.uniform(0.6, 1.3), 2)))
    if path == "fp8":  # the mode takes prefill shapes: more than 8 routes per expert on average
        low = max(64, 8 * experts // top_k + 1)
        return _case(None, path, _log_int(rng, low, 6000), zipf=zipf, **size)
    if path == "share":
        shares = rng.choice((2, 4, 8))
        return _case(None, path, _log_int(rng, 1, 6000), shares=shares, rank=rng.randrange(shares), zipf=zipf, **size)
    if path == "panels":
        return _case(None, path, _log_int(rng, 9, 2000), dtype=rng.choice(("float32", "bfloat16")), zipf=zipf, **size)
    return _case(None, path, _log_int(rng, 1, 8000), zipf=zipf, **size)


# ---------------------------------------------------------------------------------------------- inputs
def _tables(g, count, n, k, device):
    """count experts' [n, k] e4m3fn bytes and their [n / 128, k / 128] FP32 block scales."""
    bits = torch.empty((count, n, k), dtype=torch.uint8, device=device)
    scales = torch.empty((count, n // BLOCK, k // BLOCK), dtype=torch.float32, device=device)
    some = max(1, (1 << 27) // (n * k))
    for e in range(0, count, some):
        m = min(some, count - e)
        w = torch.randn((m, n // BLOCK, BLOCK, k // BLOCK, BLOCK), generator=g, device=device).mul_(0.02)
        scale = w.abs().amax(dim=(2, 4)) / 448.0
        w.div_(scale[:, :, None, :, None]).clamp_(-448.0, 448.0)
        bits[e : e + m] = w.to(torch.float8_e4m3fn).view(torch.uint8).reshape(m, n, k)
        scales[e : e + m] = scale
    return bits, scales


def _logits(case, g, device):
    logits = torch.randn((case["tokens"], case["experts"]), generator=g, device=device)
    if case["zipf"]:
        ranks = torch.arange(1, case["experts"] + 1, dtype=torch.float64)
        weight = ranks ** -case["zipf"]
        logits += torch.log(weight / weight.sum()).float().to(device)
    return logits


def _bias(case, g, device):
    return torch.randn((case["experts"],), generator=g, device=device) * (0.0 if case["zipf"] else 0.05)


def _select(logits, bias, top_k):
    """The noaux_tc routing of the logits: the k best of sigmoid + bias, weights the sigmoids over their sum."""
    scores = torch.sigmoid(logits)
    ids = torch.sort(scores + bias, dim=1, descending=True, stable=True).indices[:, :top_k]
    chosen = torch.gather(scores, 1, ids)
    return ids, chosen / chosen.sum(dim=1, keepdim=True)


def _inputs(case, seed, device):
    """Every path's inputs from the seed alone, in plain torch."""
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    h, i, e = case["hidden"], case["inter"], case["experts"]
    d = {}
    if case["path"] == "projection":
        d["x"] = torch.randn((case["tokens"], h), generator=g, device=device).to(torch.bfloat16)
        d["ids"] = torch.randint(0, e, (case["tokens"],), generator=g, device=device).to(torch.int32)
        d["tables"] = [_tables(g, e, i, h, device) for _ in range(case["tables"])]
        return d
    d["x"] = torch.randn((case["tokens"], h), generator=g, device=device).to(torch.bfloat16)
    d["logits"] = _logits(case, g, device)
    d["bias"] = _bias(case, g, device)
    ids, weights = _select(d["logits"], d["bias"], case["top_k"])
    d["ids"], d["weights"] = ids.to(torch.int32).contiguous(), weights.contiguous()
    own = e // case.get("shares", 1)
    d["gate"], d["up"], d["down"] = (_tables(g, own, i, h, device), _tables(g, own, i, h, device),
                                     _tables(g, own, h, i, device))
    if case["path"] in ("decode", "layer", "logits"):
        d["shared"] = tuple((torch.randn(s, generator=g, device=device) * 0.02).to(torch.bfloat16)
                            for s in ((i, h), (i, h), (h, i)))
    return d


def prepare(case, seed):
    d = _inputs(case, seed, torch.device("cuda"))
    path = case["path"]
    if path == "projection":
        d["owned"] = torch.ones(case["tokens"], dtype=torch.bool, device=d["x"].device)
        d["weights"] = tuple(d["tables"])
    elif path == "panels":
        d["offset"] = torch.zeros((), dtype=torch.int32, device=d["x"].device)
    else:
        d["experts"] = (*d["gate"], *d["up"], *d["down"])
    d["case"] = case
    d["contract"] = single_gpu_contract(hidden_size=case["hidden"], intermediate_size=case["inter"],
                                        num_experts=case["experts"], top_k=case["top_k"],
                                        routed_scaling_factor=ROUTED_SCALE)
    return d


# ---------------------------------------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    path = case["path"]
    if path == "decode":
        return moe_mlp_from_router_logits(s["x"], s["logits"], s["bias"], *s["experts"], contract=s["contract"],
                                          shared_bf16=s["shared"])
    if path == "layer":
        return prefill_moe_from_routes(s["x"], s["ids"], s["weights"], *s["experts"], *s["shared"],
                                       contract=s["contract"])
    if path == "logits":
        return prefill_moe_from_router_logits(s["x"], s["logits"], s["bias"], *s["experts"], *s["shared"],
                                              contract=s["contract"])
    if path == "fp8":
        return routed_experts(s["x"], s["ids"], s["weights"], *s["experts"], activations="float8_e4m3fn")
    if path == "share":
        own = case["experts"] // case["shares"]
        return routed_experts_share(s["x"], s["ids"], s["weights"], *s["experts"], num_experts=case["experts"],
                                    expert_offset=case["rank"] * own)
    if path == "projection":
        return fp8_routed_projection(s["x"], s["weights"], s["ids"], s["owned"],
                                     result_dtype=getattr(torch, case["dtype"]))
    routes = group_prefill_routes(s["ids"], num_experts=case["experts"])
    rows = gather_prefill_route_rows(s["x"], routes, top_k=case["top_k"])
    panels = build_expert_panels(routes.group_sizes, s["offset"], rows=rows.shape[0], local_groups=case["experts"])
    gate, _ = prefill_panel_fp8_matmul(rows, *s["gate"], panels, result_dtype=torch.bfloat16)
    up, _ = prefill_panel_fp8_matmul(rows, *s["up"], panels, result_dtype=torch.bfloat16)
    down, valid = prefill_panel_fp8_matmul(swiglu_bf16(gate, up), *s["down"], panels,
                                           result_dtype=getattr(torch, case["dtype"]))
    return restore_prefill_route_rows(down, routes, top_k=case["top_k"]), routes.valid, valid


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _distinct(case):
    """Experts (of this GPU's) that a case's routes select, and their routes: one drawing of its routing."""
    g = torch.Generator().manual_seed(1)
    e, k = case["experts"], case["top_k"]
    if case["path"] == "projection":
        return int(torch.randint(0, e, (case["tokens"],), generator=g).unique().numel()), case["tokens"]
    ids, _ = _select(_logits(case, g, "cpu"), _bias(case, g, "cpu"), k)
    ids = ids.reshape(-1)
    if case["path"] == "share":
        own = e // case["shares"]
        ids = ids[(ids >= case["rank"] * own) & (ids < (case["rank"] + 1) * own)]
    return int(ids.unique().numel()), int(ids.numel())


def work(case):
    t, h, i, e, k = (case[n] for n in ("tokens", "hidden", "inter", "experts", "top_k"))
    path = case["path"]
    experts, routes = _distinct(case)
    table = h * i + (h // BLOCK) * (i // BLOCK) * 4
    if path == "projection":
        n = case["tables"]
        out = 4 if case["dtype"] == "float32" else 2
        return {"bytes": experts * n * table + t * h * 2 + t * 5 + t * n * i * out, "flops": 2 * t * n * h * i}
    nbytes = experts * 3 * table + t * h * 2 + t * k * 8 + 1
    flops = 6 * routes * h * i
    if path == "share":
        nbytes += t * h * 4
    elif path == "panels":
        nbytes += t * k * h * (4 if case["dtype"] == "float32" else 2) - t * k * 4
    else:
        nbytes += t * h * 2
    if path in ("decode", "logits"):
        nbytes += t * e * 4 + e * 4
    if path in ("decode", "layer", "logits"):
        nbytes += 3 * h * i * 2
        flops += 6 * t * h * i
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """From what the outputs were measured to be off from exact()'s: 5e-3 (bf16 results of several bf16 roundings),
    2e-2 (FP8 mode: codes of the SwiGLU rows that fall on the other side of a rounding boundary), 2.3e-7 (FP32 sums)."""
    path = case["path"]
    if path == "projection" and case["dtype"] == "float32":
        return {"rel": 1e-6, "max": 2e-5}
    if path == "fp8":
        return {"rel": 3e-2, "max": 0.5}
    return {"rel": 1.2e-2, "max": 0.2, "differ": 1e-4}


# ---------------------------------------------------------------------------------------------- the same in 64 bits
def _decoded(table, e, fp8=False):
    """Expert e's weights as the projections define them: bf16(e4m3 * scale), in the FP8 mode e4m3 * scale."""
    bits, scale = table
    n, k = bits.shape[1:]
    w = bits[e].view(torch.float8_e4m3fn).to(torch.float64 if fp8 else torch.float32)
    w = w.view(n // BLOCK, BLOCK, k // BLOCK, BLOCK) * scale[e][:, None, :, None].to(w.dtype)
    return (w if fp8 else w.to(torch.bfloat16)).reshape(n, k).double()


def _quantised(x):
    """The FP8 mode's activations: e4m3 times amax / 448 per row and block of 128."""
    blocks = x.float().reshape(x.shape[0], -1, BLOCK)
    amax = blocks.abs().amax(dim=2, keepdim=True)
    scale = torch.where(amax > 0, amax / 448.0, torch.ones_like(amax))
    codes = (blocks / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return (codes.double() * scale.double()).reshape(x.shape)


def _swiglu(g, u):
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    device = torch.device("cuda")
    d = _inputs(case, seed, device)
    path = case["path"]
    x, ids = d["x"].double(), d["ids"].long()
    if path == "projection":
        out = torch.empty((case["tokens"], case["tables"], case["inter"]), dtype=torch.float64, device=device)
        for e in ids.unique().tolist():
            mine = (ids == e).nonzero().squeeze(1)
            for t, table in enumerate(d["tables"]):
                out[mine, t] = x[mine] @ _decoded(table, e).t()
        return out
    weights = d["weights"].double()
    if path in ("decode", "logits"):
        ids, weights = _select(d["logits"].double(), d["bias"].double(), case["top_k"])
    own = case["experts"] // case.get("shares", 1)
    offset = case.get("rank", 0) * own
    quantise = path == "fp8"
    if quantise:
        x = _quantised(d["x"])
    flat = ids.reshape(-1)
    count = flat.numel() if path == "panels" else case["tokens"]
    out = torch.zeros((count, case["hidden"]), dtype=torch.float64, device=device)
    for e in flat.unique().tolist():
        if not offset <= e < offset + own:
            continue
        mine = (flat == e).nonzero().squeeze(1)
        token = mine // case["top_k"]
        act = _swiglu(x[token] @ _decoded(d["gate"], e - offset, quantise).t(),
                      x[token] @ _decoded(d["up"], e - offset, quantise).t())
        if quantise:
            act = _quantised(act.to(torch.bfloat16))
        y = act @ _decoded(d["down"], e - offset, quantise).t()
        if path == "panels":
            out[mine] = y
        else:
            out.index_add_(0, token, y * weights.reshape(-1)[mine, None])
    if path == "panels":
        return out.reshape(case["tokens"], case["top_k"], case["hidden"]), None, None
    if path in ("fp8", "share"):
        return out, None
    gate, up, down = (t.double() for t in d["shared"])
    out = out * ROUTED_SCALE + _swiglu(d["x"].double() @ gate.t(), d["x"].double() @ up.t()) @ down.t()
    if path == "layer":
        return out, None
    return (out, None, weights) if path == "decode" else (out, None, weights, None)

