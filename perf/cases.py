"""What a user of nv4 runs, as cases that can be timed and compared.

A case is a dict of plain values; ``prepare`` makes its inputs and the modules
or captured graph that a program keeps, ``run`` is one pass through the
public entry points, ``work`` its unavoidable bytes and operations,
``tolerance`` what another correct implementation may differ by, and ``exact``
the same outputs in 64 bits from plain torch.  ``listed`` are fixed points of
the ranges that ``draw`` spreads over.

Kinds (``case["kind"]``); projection sizes are ``nv4.workloads.PROJECTIONS``:

* ``w4a4``: one ``W4A4Linear`` forward on bf16 rows, weights tiled as the
  loaders leave them: 1 row up to a 4096-token prompt.
* ``w4a16``: one GPTQ ``W4A16Linear`` forward, bf16 or fp16 rows.
* ``mlp``: a W4A4 MLP block with its add+RMSNorm; decode-sized calls replay
  a graph captured once, as the runner decodes, prompts run eagerly.
* ``decode``: one layer's decode attention from raw qkv rows (q/k norm, rotary,
  KV store, paged attention), replayed from a graph.
* ``step``: ``Engine.decode`` of a small GPTQ model up to the logits: input
  staging, graph replay, LM head.
* ``attention``: causal attention of packed prompts.
* ``prompt``: one prompt through a small GPTQ model (prefill) up to its logits.

The two whole models are GPTQ ones, because INT4 activation codes make a W4A4
model no measure of its parts: one bf16 ulp on a tenth of an attention output
moves a W4A4 layer's result by 10 %, and four layers' logits by 40 %
(measured).  Its parts are the ``w4a4``, ``mlp``, ``decode`` and
``attention`` cases.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "nano-vllm-int4_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from nv4.attention import decode_workspace, paged_decode_attention_qkv, prefill_attention  # noqa: E402
from nv4.engine import Engine, qwen3_8b_config  # noqa: E402
from nv4.layers import W4A4Linear, W4A16Linear  # noqa: E402
from nv4.qwen3 import Qwen3MLP, RMSNorm, get_rope  # noqa: E402
from nv4.utils.context import reset_context, set_context  # noqa: E402
from nv4.workloads import PROJECTIONS  # noqa: E402

DEV = "cuda:0"
HIDDEN, INTER, HEADS, KV_HEADS, HEAD_DIM, VOCAB = 4096, 12288, 32, 8, 128, 151936
BLOCK = 256  # tokens per KV block, the runner's default
GRAPH_ROWS = 64  # decode batches up to this replay a captured graph
EPS = 1e-6
MAX_ROWS = 4096  # the longest prompt of the benchmark
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # One request decoding outside a graph: the smallest call, host and launch latency.
        {"name": "w4a4 o, 1 row", "kind": "w4a4", "proj": "o", "rows": 1},
        # A decode batch beyond 32 sequences, ragged.
        {"name": "w4a4 gate_up, 50 rows", "kind": "w4a4", "proj": "gate_up", "rows": 50},
        # A short prompt (or a large decode batch) through the longest K.
        {"name": "w4a4 down, 200 rows", "kind": "w4a4", "proj": "down", "rows": 200},
        # An ordinary prompt, no multiple of any tile.
        {"name": "w4a4 qkv, 777 rows", "kind": "w4a4", "proj": "qkv", "rows": 777},
        # The benchmark's prompt through the widest projection.
        {"name": "w4a4 gate_up, 4096 rows", "kind": "w4a4", "proj": "gate_up", "rows": 4096},
        # The benchmark's decode batch through the block that holds most weights.
        {"name": "mlp, 32 rows", "kind": "mlp", "rows": 32},
        # GPTQ decode batch that is no multiple of 16, long K, fp16 activations as the GPTQ benchmark has them.
        {"name": "w4a16 down, 45 rows", "kind": "w4a16", "proj": "down", "rows": 45, "dtype": "fp16"},
        # GPTQ prompt.
        {"name": "w4a16 gate_up, 300 rows", "kind": "w4a16", "proj": "gate_up", "rows": 300, "dtype": "bf16"},
        # The benchmark's decode batch past its 4096-token prompts: the KV cache is most of a step.
        {"name": "decode, 32 x 4100", "kind": "decode", "batch": 32, "context": 4100},
        # A few chats decoding to their logits.
        {"name": "step, 3 x 900", "kind": "step", "layers": 4, "batch": 3, "context": 900},
        # A 4096-token prompt's attention.
        {"name": "attention, 4096", "kind": "attention", "tokens": 4096, "sequences": 1},
        # A medium prompt through the whole prefill path.
        {"name": "prompt, 1500", "kind": "prompt", "layers": 2, "tokens": 1500},
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(("w4a4", "w4a4", "w4a4", "mlp", "w4a16", "w4a16", "decode", "step", "attention", "prompt"))
    proj = rng.choice(sorted(PROJECTIONS))
    if kind == "w4a4":
        return {"kind": kind, "proj": proj, "rows": _spread(rng, 1, MAX_ROWS)}
    if kind == "w4a16":
        return {"kind": kind, "proj": proj, "rows": _spread(rng, 1, 2048), "dtype": rng.choice(sorted(DTYPES))}
    if kind == "mlp":
        return {"kind": kind, "rows": _spread(rng, 1, 1024)}
    if kind == "decode":
        batch = _spread(rng, 1, GRAPH_ROWS)
        return {"kind": kind, "batch": batch, "context": _spread(rng, 16, min(8192, 32 * 4100 // batch))}
    if kind == "step":
        batch = _spread(rng, 1, 32)
        return {"kind": kind, "layers": rng.randint(1, 3), "batch": batch, "context": _spread(rng, 16, 2048)}
    if kind == "attention":
        return {"kind": kind, "tokens": _spread(rng, 64, MAX_ROWS), "sequences": rng.randint(1, 5)}
    return {"kind": kind, "layers": 1, "tokens": _spread(rng, 16, 2048)}


# ------------------------------------------------------------------ inputs
def _rand_bytes(shape, g):
    return torch.randint(-128, 128, shape, generator=g, device=DEV, dtype=torch.int16).to(torch.int8)


def _scales(shape, g):
    return 0.005 + 0.015 * torch.rand(shape, generator=g, device=DEV)


def _activations(rows, k, g, proj):
    """bf16 rows: normal with 1 % outlier channels of 20x, as after a norm; for
    ``down`` the heavy-tailed silu(g) * u."""
    x = torch.randn(rows, k, generator=g, device=DEV)
    if proj == "down":
        return (torch.nn.functional.silu(x) * torch.randn(rows, k, generator=g, device=DEV)).to(torch.bfloat16)
    x[:, torch.randperm(k, generator=g, device=DEV)[:k // 100]] *= 20.0
    return x.to(torch.bfloat16)


def _fill_w4a4(linear, g):
    n, k = linear.out_features, linear.in_features
    signs = torch.randint(0, 2, (k,), generator=g, device=DEV, dtype=torch.int16) * 2 - 1
    packed, scale = _rand_bytes((n, k // 2), g), _scales((n, k // 128), g).to(torch.bfloat16)
    linear.assign_quantized_(packed, scale, signs.to(torch.int8))
    return packed


def _on_device(make):
    before = torch.get_default_dtype()
    torch.set_default_dtype(torch.bfloat16)
    try:
        with torch.device(DEV):
            return make()
    finally:
        torch.set_default_dtype(before)


def _lengths(total, parts, seed):
    """``parts`` ragged lengths, at least 1 each, that sum to ``total``."""
    g = torch.Generator("cpu").manual_seed(seed)
    cuts = sorted((torch.randperm(total - 1, generator=g)[:parts - 1] + 1).tolist())
    return [b - a for a, b in zip([0] + cuts, cuts + [total])]


def _contexts(batch, context):
    """Ragged contexts, fixed by the case: the last few per cent below ``context``."""
    return [max(1, context - (7 * i) % max(1, context // 16)) for i in range(batch)]


def prepare(case, seed):
    with torch.no_grad():
        return _PREPARE[case["kind"]](case, torch.Generator(device=DEV).manual_seed(seed), seed)


def _prepare_w4a4(case, g, seed):
    n, k = PROJECTIONS[case["proj"]]
    linear = _on_device(lambda: W4A4Linear(k, n))
    packed = _fill_w4a4(linear, g)
    return {"kind": "w4a4", "module": linear, "x": _activations(case["rows"], k, g, case["proj"]), "packed": packed}


def _prepare_w4a16(case, g, seed):
    n, k = PROJECTIONS[case["proj"]]
    linear = _on_device(lambda: W4A16Linear(k, n))
    for p in (linear.qweight, linear.qzeros):
        p.copy_(torch.randint(-2**31, 2**31, p.shape, generator=g, device=DEV, dtype=torch.int64))
    linear.scales.copy_(_scales(linear.scales.shape, g))
    x = torch.randn(case["rows"], k, generator=g, device=DEV).to(DTYPES[case["dtype"]])
    return {"kind": "w4a16", "module": linear, "x": x}


def _captured(step):
    """``step`` in a graph, after a warm-up on a side stream, as the runner captures it."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    return graph, out


def _prepare_mlp(case, g, seed):
    mlp, norm = _on_device(lambda: (Qwen3MLP(HIDDEN, INTER, use_w4a4=True), RMSNorm(HIDDEN, EPS)))
    _fill_w4a4(mlp.gate_up_proj, g)
    _fill_w4a4(mlp.down_proj, g)
    norm.weight.copy_(1 + 0.1 * torch.randn(HIDDEN, generator=g, device=DEV))
    x, before = (_activations(case["rows"], HIDDEN, g, "gate_up") for _ in range(2))

    def step():  # the block adds into its residual: each pass starts from the same one
        out, residual = mlp.forward_fused(x, before.clone(), norm)
        return {"out": out, "residual": residual}

    graph, out = _captured(step) if case["rows"] <= GRAPH_ROWS else (None, None)
    return {"kind": "mlp", "step": step, "graph": graph, "out": out}


def _prepare_decode(case, g, seed):
    batch, context = case["batch"], case["context"]
    rope = get_rope(HEAD_DIM, 40960, 1_000_000.0).cos_sin_cache.to(DEV)
    norms = [(1 + 0.1 * torch.randn(HEAD_DIM, generator=g, device=DEV)).to(torch.bfloat16) for _ in range(2)]
    blocks = -(-context // BLOCK)
    caches = [torch.randn(batch * blocks, BLOCK, KV_HEADS, HEAD_DIM, generator=g, device=DEV, dtype=torch.bfloat16)
              for _ in range(2)]
    qkv = torch.randn(batch, (HEADS + 2 * KV_HEADS) * HEAD_DIM, generator=g, device=DEV).to(torch.bfloat16)
    lens = torch.tensor(_contexts(batch, context), device=DEV)
    tables = torch.randperm(batch * blocks, generator=g, device=DEV).to(torch.int32).view(batch, blocks)
    last = lens - 1
    slots = tables.gather(1, (last // BLOCK)[:, None]).view(-1) * BLOCK + (last % BLOCK).to(torch.int32)
    work_space, lens = decode_workspace(batch, HEADS, blocks * BLOCK, HEAD_DIM, DEV), lens.to(torch.int32)

    def step():
        return paged_decode_attention_qkv(qkv, HEADS, KV_HEADS, *norms, rope, last, slots, EPS, *caches, tables, lens,
                                          HEAD_DIM ** -0.5, workspace=work_space, max_context=blocks * BLOCK)

    graph, out = _captured(step)
    return {"kind": "decode", "step": step, "graph": graph, "qkv": qkv, "norms": norms, "rope": rope, "lens": lens,
            "tables": tables, "out": {"out": out, "k_cache": caches[0], "v_cache": caches[1]}}


def _engine(layers, batch, context, g, seed, graph=False):
    engine = Engine(qwen3_8b_config(layers), use_w4a4=False, use_w4a16=True, max_num_seqs=batch,
                    max_model_len=context, device=DEV, seed=seed)
    if graph:  # its warm-up writes the cache: before the cache is filled
        engine.capture(batch)
    engine.kv_cache.copy_(torch.randn(engine.kv_cache.shape, generator=g, device=DEV, dtype=torch.bfloat16))
    return engine


def _prepare_step(case, g, seed):
    batch = case["batch"]
    engine = _engine(case["layers"], batch, case["context"], g, seed, graph=True)
    tokens = torch.randint(0, VOCAB, (batch,), generator=g, device=DEV).tolist()
    return {"kind": "step", "engine": engine, "slots": list(range(batch)), "tokens": tokens,
            "lengths": _contexts(batch, case["context"]), "temperatures": torch.full((batch,), 0.6, device=DEV)}


def _prepare_attention(case, g, seed):
    t = case["tokens"]

    def rows(heads):
        return torch.randn(t, heads, HEAD_DIM, generator=g, device=DEV).to(torch.bfloat16)

    # The lengths are the case's own, so that every seed is the same work.
    return {"kind": "attention", "q": rows(HEADS), "k": rows(KV_HEADS), "v": rows(KV_HEADS),
            "lens": _lengths(t, case["sequences"], t), "scale": HEAD_DIM ** -0.5}


def _prepare_prompt(case, g, seed):
    n = case["tokens"]
    engine = _engine(case["layers"], 1, n, g, seed)
    ids = torch.randint(0, VOCAB, (n,), generator=g, device=DEV)
    return {"kind": "prompt", "engine": engine, "ids": ids, "positions": torch.arange(n, device=DEV),
            "cu": torch.tensor([0, n], dtype=torch.int32, device=DEV), "n": n,
            "slots": torch.arange(n, dtype=torch.int32, device=DEV)}


_PREPARE = {"w4a4": _prepare_w4a4, "w4a16": _prepare_w4a16, "mlp": _prepare_mlp, "decode": _prepare_decode,
            "step": _prepare_step, "attention": _prepare_attention, "prompt": _prepare_prompt}


# -------------------------------------------------------------------- runs
@torch.inference_mode()
def run(state):
    kind = state["kind"]
    if kind in ("w4a4", "w4a16"):
        return state["module"](state["x"])
    if kind in ("mlp", "decode"):
        if state["graph"] is None:
            return state["step"]()
        state["graph"].replay()
        return state["out"]
    if kind == "step":
        logits = state["engine"].decode(state["slots"], state["tokens"], state["lengths"], state["temperatures"],
                                        return_logits=True)
        return {"logits": logits, "kv_cache": state["engine"].kv_cache}
    if kind == "attention":
        return prefill_attention(state["q"], state["k"], state["v"], state["lens"], state["scale"])
    engine, n = state["engine"], state["n"]
    set_context(True, state["cu"], state["cu"], n, n, state["slots"], None, None, seqlens_q=(n,))
    logits = engine.model.compute_logits(engine.model(state["ids"], state["positions"]))
    reset_context()
    return {"logits": logits, "kv_cache": engine.kv_cache}


# ----------------------------------------------------------- work, tolerance
def _linear(proj, rows, zeros=False):
    """(bytes, operations) of one quantized projection: rows in and out in 16
    bits, 4-bit codes, 16-bit group scales (and 4-bit zero points)."""
    n, k = PROJECTIONS[proj]
    weights = n * k // 2 + 2 * n * k // 128 + (n * k // 256 if zeros else k)
    return 2 * rows * (n + k) + weights, 2 * rows * n * k


def _pairs(lens):
    return sum(n * (n + 1) // 2 for n in lens)


_KV = 4 * KV_HEADS * HEAD_DIM  # bytes of a token's key and value


def work(case):
    kind = case["kind"]
    if kind in ("w4a4", "w4a16"):
        size, flops = _linear(case["proj"], case["rows"], kind == "w4a16")
    elif kind == "mlp":  # x and the residual in, both out; what lies between the projections stays on the chip
        m = case["rows"]
        (b1, f1), (b2, f2) = _linear("gate_up", 0), _linear("down", 0)
        size, flops = b1 + b2 + 8 * m * HIDDEN, m * 2 * (3 * HIDDEN * INTER)
    elif kind == "decode":
        total = sum(_contexts(case["batch"], case["context"]))
        size = _KV * total + 2 * case["batch"] * (2 * HEADS + 2 * KV_HEADS) * HEAD_DIM
        flops = 4 * HEADS * HEAD_DIM * total
    elif kind == "attention":
        t = case["tokens"]
        size = 4 * t * (HEADS + KV_HEADS) * HEAD_DIM
        flops = 4 * HEADS * HEAD_DIM * _pairs(_lengths(t, case["sequences"], t))
    else:
        weights = sum(_linear(p, 0, True)[0] for p in PROJECTIONS)
        if kind == "step":
            rows = heads = case["batch"]
            tokens = pairs = sum(_contexts(rows, case["context"]))
        else:
            rows, heads, tokens = case["tokens"], 1, case["tokens"]
            pairs = _pairs([tokens])
        layer = sum(_linear(p, rows, True)[1] for p in PROJECTIONS) + 4 * HEADS * HEAD_DIM * pairs
        size = case["layers"] * (weights + _KV * tokens) + 2 * (VOCAB * HIDDEN + rows * HIDDEN + heads * VOCAB)
        flops = case["layers"] * layer + 2 * heads * VOCAB * HIDDEN
    return {"bytes": size, "flops": flops}


# Single operators: four times the distance from the 64-bit result, which is
# the rounding of a 16-bit result (1.7e-3 in bf16) and, for GPTQ, of each
# dequantized weight (2.9e-3) or, for attention, of q, k and the probabilities
# (2e-3, 3.6e-3).  Whole models: four times what they moved by with fp32
# attention and unrounded GPTQ weights in place of the kernels (logits 4e-3
# .. 5e-3, the second layer's keys and values 7e-3).  The MLP quantizes
# its first projection's bf16 results again, so a few that round the other way
# come out as other INT4 codes.
_TOLERANCE = {"w4a4": {"rel": 7e-3}, "mlp": {"rel": 2e-2}, "w4a16": {"rel": 1.2e-2}, "attention": {"rel": 8e-3},
              "decode": {"rel": 1.4e-2}, "step": {"rel": 2e-2}, "prompt": {"rel": 3e-2}}


def tolerance(case):
    return _TOLERANCE[case["kind"]]


# ------------------------------------------------------------- 64-bit results
def _hadamard(x, bits):
    """Sylvester transform of the last axis (2^bits long), unnormalised."""
    shape = x.shape
    for b in range(bits):
        x = x.view(*shape[:-1], -1, 2, 1 << b)
        x = torch.stack((x[..., 0, :] + x[..., 1, :], x[..., 0, :] - x[..., 1, :]), dim=-2)
    return x.reshape(shape)


def _rht(x, signs):
    """Signs, then the Hadamard matrix of order K: Sylvester, for K = 12288
    Paley's matrix of order 12 over chunks of 1024."""
    x = x.double() * signs.double()
    m, k = x.shape
    if k == 4096:
        return _hadamard(x, 12) / 64
    squares = {1, 3, 4, 5, 9}
    h12 = torch.tensor([[1.0 if s == 0 or d == 0 or (d - s) % 11 in squares else -1.0 for d in range(12)]
                        for s in range(12)], dtype=torch.float64, device=x.device)
    x = _hadamard(x.view(m, 12, 1024), 10) / 32
    x = x.permute(0, 2, 1).reshape(-1, 12) @ h12 / math.sqrt(12.0)
    return x.view(m, 1024, 12).permute(0, 2, 1).reshape(m, k)


def _nibbles(packed):
    """int8 [R, C] of two codes each, low nibble first -> float64 [R, 2 C]."""
    p = packed.to(torch.int16) & 255
    q = torch.stack((p & 15, p >> 4), dim=-1).flatten(-2)
    return (q - 16 * (q > 7)).double()


def _exact_w4a4(s):
    linear, x = s["module"], s["x"]
    m, k = x.shape
    rows = _rht(x, linear.signs).view(m, k // 128, 128)
    top = rows.abs().amax(dim=-1, keepdim=True)
    scale = torch.where(top > 0, top * 0.9 / 7, torch.ones_like(top)).float().to(torch.bfloat16).double()
    a = ((rows / scale).round().clamp(-7, 7) * scale).view(m, k)
    out = torch.empty(m, linear.out_features, dtype=torch.float64, device=x.device)
    for n in range(0, linear.out_features, 4096):
        w = _nibbles(s["packed"][n:n + 4096]).view(-1, k // 128, 128)
        w *= linear.weight_scale[n:n + 4096].double()[..., None]
        out[:, n:n + 4096] = a @ w.view(-1, k).t().contiguous()
    return out


def _exact_w4a16(s):
    linear, x = s["module"], s["x"].double()
    k, n = linear.in_features, linear.out_features
    by = 4 * torch.arange(8, device=DEV, dtype=torch.int32)
    z = ((linear.qzeros[:, :, None] >> by) & 15).reshape(k // 128, n) + 1
    q = ((linear.qweight[:, None, :] >> by[:, None]) & 15).reshape(k // 128, 128, n)
    out = torch.zeros(x.shape[0], n, dtype=torch.float64, device=x.device)
    for i in range(k // 128):
        out += x[:, 128 * i:128 * i + 128].contiguous() @ ((q[i] - z[i]).double() * linear.scales[i].double())
    return out


def _exact_attention(s):
    q, k, v = (s[x].double() for x in "qkv")
    out, at = torch.empty_like(q), 0
    for n in s["lens"]:
        hidden = torch.ones(n, n, dtype=torch.bool, device=DEV).triu(1)
        for h in range(HEADS):
            kv = h // (HEADS // KV_HEADS)
            p = q[at:at + n, h].contiguous() @ k[at:at + n, kv].t().contiguous() * s["scale"]
            out[at:at + n, h] = p.masked_fill_(hidden, -math.inf).softmax(dim=-1) @ v[at:at + n, kv].contiguous()
        at += n
    return out


def _exact_decode(s):
    heads = s["qkv"].double().view(-1, HEADS + 2 * KV_HEADS, HEAD_DIM)
    cos, sin = s["rope"].view(-1, HEAD_DIM)[s["lens"].long() - 1].double()[:, None, :].chunk(2, dim=-1)

    def rotated(x, w):
        x = x * (x.square().mean(dim=-1, keepdim=True) + EPS).rsqrt() * w.double()
        a, b = x.chunk(2, dim=-1)
        return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)

    q = rotated(heads[:, :HEADS], s["norms"][0])
    keys = rotated(heads[:, HEADS:HEADS + KV_HEADS], s["norms"][1])
    out = torch.empty_like(q)
    for i, n in enumerate(s["lens"].tolist()):
        k, v = (s["out"][c][s["tables"][i].long()].reshape(-1, KV_HEADS, HEAD_DIM)[:n].double()
                for c in ("k_cache", "v_cache"))
        k[-1], v[-1] = keys[i], heads[i, HEADS + KV_HEADS:]
        for h in range(KV_HEADS):
            at = slice(h * (HEADS // KV_HEADS), (h + 1) * (HEADS // KV_HEADS))
            p = (q[i, at] @ k[:, h].t().contiguous() * HEAD_DIM ** -0.5).softmax(dim=-1)
            out[i, at] = p @ v[:, h].contiguous()
    return {"out": out, "k_cache": None, "v_cache": None}


@torch.no_grad()
def exact(case, seed):
    """None for the MLP and for whole models, whose 16-bit roundings between
    operators are part of what they compute."""
    of = {"w4a4": _exact_w4a4, "w4a16": _exact_w4a16, "attention": _exact_attention,
          "decode": _exact_decode}.get(case["kind"])
    return None if of is None else of(prepare(case, seed))
