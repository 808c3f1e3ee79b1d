"""Performance cases of the verify-step operators: what is timed, over which
sizes, and how far another correct implementation may be off.

A case is a dict of plain values with a ``kind``:

  layer    the packed linears of one transformer layer (qkv, o, gate/up as one
           group, down), bound through PackedLinearOperators: one captured
           graph for decode and verify sizes, eager launches for prefill
  head     the packed lm_head alone
  verify   the whole verify step of a small model: lm_head, then the fused
           acceptance, in one captured graph
  accept   the fused acceptance over given target logits
  greedy   one replay of the captured greedy sampler over given logits
  moe      a routed-expert block: router, compaction, gate/up, down
  embed    the packed embedding lookup

Weights are random Cubic payloads whose codes are those of normally
distributed weights (scale near three standard deviations), activations are
N(0, 1), logits N(0, 3).
"""
from __future__ import annotations

import math

import torch

from cubic_serve_amd import greedy, linear, moe, quantization as qz, sampling

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
BLOCK_M = 32  # route slots per padded block, the operator's default


def listed() -> list[dict]:
    return [
        # smallest call: one sequence with one draft on a 32768-token head
        {"name": "verify_small_m2", "kind": "verify", "hidden": 2048, "vocab": 32768, "bits": 4,
         "group": 128, "c": 1, "depth": 1},
        # single-sequence decode of a Llama-3-70B-shaped layer: the weight stream
        {"name": "layer70b_w4_m1", "kind": "layer", "hidden": 8192, "qkv": 10240, "inter": 28672,
         "bits": 4, "group": 128, "m": 1, "layers": 1, "dtype": "bf16"},
        # a few sequences (4 x (1 draft + 1)) on the same layer
        {"name": "layer70b_w4_m8", "kind": "layer", "hidden": 8192, "qkv": 10240, "inter": 28672,
         "bits": 4, "group": 128, "m": 8, "layers": 1, "dtype": "bf16"},
        # the same at 6 bits, the accuracy-first width
        {"name": "layer70b_w6_m8", "kind": "layer", "hidden": 8192, "qkv": 10240, "inter": 28672,
         "bits": 6, "group": 128, "m": 8, "layers": 1, "dtype": "bf16"},
        # the benchmark's verify step: batch 32 x (1 draft + 1), Qwen3-8B-shaped layers
        {"name": "layers8b_w4_m64", "kind": "layer", "hidden": 4096, "qkv": 6144, "inter": 12288,
         "bits": 4, "group": 128, "m": 64, "layers": 4, "dtype": "bf16"},
        # prompt processing, a full chunk
        {"name": "layer8b_w4_m2048", "kind": "layer", "hidden": 4096, "qkv": 6144, "inter": 12288,
         "bits": 4, "group": 128, "m": 2048, "layers": 1, "dtype": "bf16"},
        # the ragged last chunk of a prompt, 8-bit weights, fp16 activations
        {"name": "layer8b_w8_m333_f16", "kind": "layer", "hidden": 4096, "qkv": 6144, "inter": 12288,
         "bits": 8, "group": 128, "m": 333, "layers": 1, "dtype": "fp16"},
        # the quantized head of the verify step
        {"name": "head8b_w4_m64", "kind": "head", "hidden": 4096, "vocab": 151936, "bits": 4,
         "group": 128, "m": 64, "dtype": "bf16"},
        # stochastic acceptance: 64 sequences x 3 drafts, T 0.7, top-p 0.9, top-k 20
        {"name": "accept_c64_k3", "kind": "accept", "vocab": 151936, "c": 64, "depth": 3,
         "temperature": 0.7, "hit": 0.7},
        # greedy sampling of plain decode, 64 rows
        {"name": "greedy_r64", "kind": "greedy", "vocab": 151936, "rows": 64},
        # routed experts: 256 tokens, 128 experts, top-8
        {"name": "moe_t256", "kind": "moe", "hidden": 2048, "inter": 768, "experts": 128, "top_k": 8,
         "tokens": 256, "bits": 4, "group": 128},
        # prompt token lookup
        {"name": "embed_t4096", "kind": "embed", "hidden": 4096, "vocab": 151936, "bits": 4,
         "group": 128, "tokens": 4096, "dtype": "bf16"},
    ]


# ---------------------------------------------------------------------------
# drawn cases
# ---------------------------------------------------------------------------
def _log(rng, low: int, high: int, step: int = 1) -> int:
    """A multiple of ``step``, spread over the logarithm of [low, high]."""
    value = math.exp(rng.uniform(math.log(low), math.log(high)))
    return max(low, min(high, int(round(value / step)) * step))


def draw(rng) -> dict:
    kind = rng.choices(("layer", "head", "verify", "accept", "greedy", "moe", "embed"),
                       (8, 2, 1, 2, 1, 2, 1))[0]
    bits = rng.choices((1, 2, 3, 4, 5, 6, 7, 8), (1, 3, 3, 10, 1, 3, 1, 3))[0]
    group = rng.choices((128, 64, 32), (8, 1, 1))[0]
    dtype = rng.choices(("bf16", "fp16"), (3, 1))[0]
    if kind == "layer":
        hidden = _log(rng, 1024, 8192, 128)
        inter = min(28672, _log(rng, 2 * hidden, 4 * hidden, 128))
        qkv = _log(rng, hidden, 2 * hidden, 64)
        weights = hidden * (hidden + qkv + 3 * inter)
        # cost bound: the largest listed prefill is about 0.8 TFLOP
        most = max(8, min(2048, int(1.2e11 // weights)))
        return {"kind": "layer", "hidden": hidden, "qkv": qkv, "inter": inter, "bits": bits,
                "group": group, "m": _log(rng, 1, most), "layers": 1, "dtype": dtype}
    if kind == "head":
        return {"kind": "head", "hidden": _log(rng, 1024, 5120, 128), "vocab": _log(rng, 16000, 151936),
                "bits": bits, "group": group, "m": _log(rng, 1, 128), "dtype": dtype}
    if kind == "verify":
        depth = rng.randint(1, 3)
        return {"kind": "verify", "hidden": _log(rng, 1024, 4096, 128), "vocab": _log(rng, 16000, 64000),
                "bits": bits, "group": group, "c": _log(rng, 1, 16), "depth": depth}
    if kind == "accept":
        return {"kind": "accept", "vocab": _log(rng, 16000, 151936), "c": _log(rng, 1, 64),
                "depth": rng.randint(1, 3), "temperature": rng.choice((0.0, 0.7, 1.0)), "hit": 0.7}
    if kind == "greedy":
        return {"kind": "greedy", "vocab": _log(rng, 16000, 151936), "rows": _log(rng, 1, 256)}
    if kind == "moe":
        return {"kind": "moe", "hidden": _log(rng, 1024, 4096, 128), "inter": _log(rng, 512, 1536, 128),
                "experts": rng.choice((16, 32, 64)), "top_k": rng.choice((2, 4, 8)),
                "tokens": _log(rng, 1, 512), "bits": bits, "group": group}
    return {"kind": "embed", "hidden": _log(rng, 1024, 8192, 128), "vocab": _log(rng, 16000, 151936),
            "bits": bits, "group": group, "tokens": _log(rng, 1, 16384), "dtype": dtype}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _device() -> torch.device:
    return torch.device("cuda:0")


def _generator(seed: int) -> torch.Generator:
    return torch.Generator(device=_device()).manual_seed(seed)


def _payload(gen, n: int, k: int, bits: int, group: int) -> qz.QuantizedMatrix:
    """A random [n, k] Cubic matrix (format 0), k a multiple of 8: eight codes
    make ``bits`` bytes, assembled in a 64-bit word."""
    dev = _device()
    top = (1 << (bits - 1)) - 1
    packed = torch.empty((n, k // 8 * bits), dtype=torch.uint8, device=dev)
    shifts = torch.arange(8, device=dev, dtype=torch.int64) * bits
    rows = max(1, (1 << 26) // k)
    for r in range(0, n, rows):
        count = min(rows, n - r)
        v = torch.randn((count, k), generator=gen, device=dev)
        if bits == 1:
            raw = (v > 0).to(torch.int64)
        else:
            raw = (v * (top / 3.0)).round_().clamp_(-top, top).to(torch.int64) & ((1 << bits) - 1)
        words = (raw.view(count, k // 8, 8) << shifts).sum(-1, dtype=torch.int64)
        packed[r:r + count] = words.view(torch.uint8).view(count, k // 8, 8)[:, :, :bits].reshape(count, -1)
    groups = (n, -(-k // group))
    curves = torch.tensor(qz.CURVES, device=dev)
    pick = curves[torch.randint(0, len(qz.CURVES), groups, generator=gen, device=dev)]
    payload = {"weight_packed": packed,
               "weight_scale": torch.rand(groups, generator=gen, device=dev) * 0.02 + 0.05,
               "weight_a": pick[..., 0].half().contiguous(), "weight_b": pick[..., 1].half().contiguous()}
    return qz.QuantizedMatrix(payload, qz.QuantizationScheme(qz.CUBIC_FORMAT, bits, group), (n, k))


def _normal(gen, shape, dtype) -> torch.Tensor:
    return torch.randn(shape, generator=gen, device=_device()).to(dtype)


def _captured(launch) -> torch.cuda.CUDAGraph:
    """A graph of ``launch``, as a serving loop captures its step."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        launch()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        launch()
    torch.cuda.synchronize()
    return graph


GRAPH_ROWS = 128  # decode and verify batches are captured, prompts run eagerly


def _layer_inputs(case: dict, gen):
    """Per layer: the activations of hidden and intermediate width, then the
    five matrices."""
    dtype, h, i = DTYPES[case["dtype"]], case["hidden"], case["inter"]
    for _ in range(case["layers"]):
        x = _normal(gen, (case["m"], h), dtype)
        x_down = _normal(gen, (case["m"], i), dtype)
        weights = [_payload(gen, n, k, case["bits"], case["group"]) for n, k in
                   ((case["qkv"], h), (h, h), (i, h), (i, h), (h, i))]
        yield x, x_down, weights


def _prepare_layer(case: dict, seed: int) -> dict:
    ops = linear.PackedLinearOperators()
    bindings, outputs, keep = [], [], []
    for x, x_down, (qkv, o, gate, up, down) in _layer_inputs(case, _generator(seed)):
        ys = [torch.empty((x.shape[0], w.shape[0]), dtype=x.dtype, device=x.device)
              for w in (qkv, o, gate, up, down)]
        bindings += [ops.bind_linear(x, qkv, ys[0]), ops.bind_linear(x, o, ys[1]),
                     ops.bind_linear_group(x, (gate, up), ys[2:4]), ops.bind_linear(x_down, down, ys[4])]
        outputs += ys
        keep += [x, x_down]
    state = {"ops": ops, "bindings": bindings, "outputs": outputs, "keep": keep, "graph": None}
    if case["m"] <= GRAPH_ROWS:
        state["graph"] = _captured(lambda: [b.launch() for b in bindings])
    return state


def _prepare_head(case: dict, seed: int) -> dict:
    gen = _generator(seed)
    x = _normal(gen, (case["m"], case["hidden"]), DTYPES[case["dtype"]])
    weight = _payload(gen, case["vocab"], case["hidden"], case["bits"], case["group"])
    y = torch.empty((case["m"], case["vocab"]), dtype=x.dtype, device=x.device)
    ops = linear.PackedLinearOperators()
    return {"ops": ops, "bindings": [ops.bind_linear(x, weight, y)], "outputs": [y], "keep": [x],
            "graph": None}


def _accept_plan(logits, gen, c: int, depth: int, temperature: float, drafts, q_scores, q_ids):
    dev = logits.device
    shape = (depth, c)
    return sampling.MTPVerifyPlan(
        logits=logits, q_scores=q_scores, q_token_ids=q_ids, draft_tokens=drafts,
        temperatures=torch.full(shape, temperature, device=dev),
        top_ps=torch.full(shape, 0.9 if temperature else 1.0, device=dev),
        top_ks=torch.full(shape, 20, dtype=torch.int64, device=dev),
        seeds=torch.randint(0, 2**40, shape, generator=gen, device=dev),
        ordinals=torch.randint(0, 10000, shape, generator=gen, device=dev),
        uniforms=torch.rand((depth, c, 2), generator=gen, device=dev))


def _verify_inputs(case: dict, seed: int):
    """Head, activations that point at one token each (a trained model's top
    logit stands clear of the rest) and drafts that mostly hit it."""
    gen = _generator(seed)
    dev = _device()
    c, depth, vocab = case["c"], case["depth"], case["vocab"]
    rows = c * (depth + 1)
    weight = _payload(gen, vocab, case["hidden"], case["bits"], case["group"])
    target = torch.randint(0, vocab, (rows,), generator=gen, device=dev)
    x = torch.randn((rows, case["hidden"]), generator=gen, device=dev)
    x = (x + 30.0 * _decode(weight, torch.float32, target).float()).to(torch.bfloat16)
    hit = torch.rand((rows,), generator=gen, device=dev) < 0.7
    other = (target + 1 + torch.randint(0, vocab - 1, (rows,), generator=gen, device=dev)) % vocab
    drafts = torch.where(hit, target, other).view(c, depth + 1)[:, :depth].t().contiguous()
    return gen, weight, x, drafts


def _prepare_verify(case: dict, seed: int) -> dict:
    gen, weight, x, drafts = _verify_inputs(case, seed)
    dev = x.device
    c, depth = case["c"], case["depth"]
    logits = torch.empty((x.shape[0], case["vocab"]), dtype=x.dtype, device=dev)
    q_scores = torch.full((depth, c, 20), float("nan"), dtype=torch.bfloat16, device=dev)
    q_scores[:, :, 0] = 1.0
    q_ids = torch.full((depth, c, 20), -1, dtype=torch.int64, device=dev)
    q_ids[:, :, 0] = drafts
    ops = linear.PackedLinearOperators()
    head = ops.bind_linear(x, weight, logits)
    plan = _accept_plan(logits, gen, c, depth, 0.0, drafts, q_scores, q_ids)
    graph = _captured(lambda: (head.launch(), plan.launch()))
    return {"ops": ops, "head": head, "plan": plan, "graph": graph,
            "outputs": [logits, plan.decisions, plan.merged, plan.emitted]}


def _accept_inputs(case: dict, seed: int):
    """Target logits, and the draft's logits near them; a draft token is the
    draft's own best with the hit rate, else one of its next few."""
    gen = _generator(seed)
    dev = _device()
    c, depth, vocab = case["c"], case["depth"], case["vocab"]
    target = (torch.randn((c * (depth + 1), vocab), generator=gen, device=dev) * 3).to(torch.bfloat16)
    q_scores = torch.empty((depth, c, 20), dtype=torch.bfloat16, device=dev)
    q_ids = torch.empty((depth, c, 20), dtype=torch.int64, device=dev)
    for d in range(depth):
        q = target[d::depth + 1].float() + torch.randn((c, vocab), generator=gen, device=dev)
        # distinct scores from 20 to 1, order fixed by a stable sort
        _, order = torch.sort(q.to(torch.bfloat16).float(), dim=-1, descending=True, stable=True)
        q_ids[d] = order[:, :20]
        q_scores[d] = torch.gather(q, 1, q_ids[d]).to(torch.bfloat16)
    slot = torch.where(torch.rand((depth, c), generator=gen, device=dev) < case["hit"], 0,
                       torch.randint(1, 5, (depth, c), generator=gen, device=dev))
    drafts = torch.gather(q_ids, 2, slot[..., None])[..., 0].contiguous()
    return gen, target, q_scores, q_ids, drafts


def _prepare_accept(case: dict, seed: int) -> dict:
    gen, target, q_scores, q_ids, drafts = _accept_inputs(case, seed)
    plan = _accept_plan(target, gen, case["c"], case["depth"], case["temperature"], drafts, q_scores, q_ids)
    return {"plan": plan, "outputs": [plan.candidate_scores, plan.candidate_ids, plan.decisions,
                                      plan.merged, plan.emitted]}


def _greedy_logits(case: dict, seed: int):
    gen = _generator(seed)
    logits = torch.randn((case["rows"], case["vocab"]), generator=gen, device=_device()) * 3
    return logits.to(torch.bfloat16)


def _prepare_greedy(case: dict, seed: int) -> dict:
    logits = _greedy_logits(case, seed)
    dev, rows = logits.device, case["rows"]
    params = greedy.ShardedSamplingParameters(
        torch.zeros(rows, device=dev), torch.full((rows,), 20, dtype=torch.int64, device=dev),
        torch.full((rows,), 0.95, device=dev), 20, torch.ones(rows, dtype=torch.int64, device=dev),
        torch.zeros(rows, dtype=torch.int64, device=dev))
    workspace = sampling.ShardedSamplingWorkspace(
        torch.empty((rows, 20), dtype=torch.bfloat16, device=dev),
        torch.empty((rows, 20), dtype=torch.int64, device=dev), None, None)
    sampler = greedy.CapturedGreedySampler(
        local_logits=logits, true_vocab_size=case["vocab"],
        token_ids=torch.empty(rows, dtype=torch.int64, device=dev), parameters=params,
        workspace=workspace, root_valid=torch.empty(rows, dtype=torch.bool, device=dev))
    return {"sampler": sampler, "rows": rows, "valid": torch.zeros((), dtype=torch.bool, device=dev)}


def _moe_inputs(case: dict, seed: int):
    gen = _generator(seed)
    e, h, i, t = case["experts"], case["hidden"], case["inter"], case["tokens"]
    router = _normal(gen, (t, e), torch.bfloat16)
    x = _normal(gen, (t, h), torch.bfloat16)
    x_down = _normal(gen, (t * case["top_k"], i), torch.bfloat16)
    stacked = [_payload(gen, e * n, k, case["bits"], case["group"]) for n, k in ((i, h), (i, h), (h, i))]
    return router, x, x_down, stacked


def _prepare_moe(case: dict, seed: int) -> dict:
    router, x, x_down, (gate, up, down) = _moe_inputs(case, seed)
    dev, e, t, top_k = x.device, case["experts"], case["tokens"], case["top_k"]
    split = lambda w: tuple(w.rows(j * (w.shape[0] // e), (j + 1) * (w.shape[0] // e)) for j in range(e))
    routing = moe.MoERouting(router, torch.ones(t, dtype=torch.int32, device=dev),
                             torch.tensor([t], dtype=torch.int32, device=dev), top_k=top_k, block_m=BLOCK_M)
    h = torch.empty((t * top_k, 2 * case["inter"]), dtype=x.dtype, device=dev)
    y = torch.empty((t * top_k, case["hidden"]), dtype=x.dtype, device=dev)
    ops = linear.PackedLinearOperators()
    gate_up = moe.bind_grouped(ops, x, split(gate), split(up), h, routing.rows, top_k)[1]
    routed = moe.bind_routed(ops, x_down, split(down), y, routing.rows)[1]
    return {"ops": ops, "routing": routing, "bindings": [gate_up, routed],
            "outputs": [routing.route_ids, routing.route_weights, h, y]}


def _embed_inputs(case: dict, seed: int):
    gen = _generator(seed)
    table = _payload(gen, case["vocab"], case["hidden"], case["bits"], case["group"])
    ids = torch.randint(0, case["vocab"], (case["tokens"],), generator=gen, device=_device())
    return table, ids


def _prepare_embed(case: dict, seed: int) -> dict:
    table, ids = _embed_inputs(case, seed)
    y = torch.empty((case["tokens"], case["hidden"]), dtype=DTYPES[case["dtype"]], device=ids.device)
    ops = linear.PackedLinearOperators()
    return {"ops": ops, "bindings": [ops.bind_embedding(ids, table, y)], "outputs": [y], "graph": None}


def prepare(case: dict, seed: int) -> dict:
    state = {"layer": _prepare_layer, "head": _prepare_head, "verify": _prepare_verify,
             "accept": _prepare_accept, "greedy": _prepare_greedy, "moe": _prepare_moe,
             "embed": _prepare_embed}[case["kind"]](case, seed)
    state["kind"] = case["kind"]
    return state


def run(state: dict):
    kind = state["kind"]
    if kind == "greedy":
        tokens = state["sampler"].replay(state["rows"], validity_out=state["valid"])
        return [tokens, state["valid"]]
    if kind == "accept":
        state["plan"].launch()
    elif kind == "moe":
        state["routing"].launch()
        for binding in state["bindings"]:
            binding.launch()
    elif state["graph"] is not None:
        state["graph"].replay()
    else:
        for binding in state["bindings"]:
            binding.launch()
    return state["outputs"]


# ---------------------------------------------------------------------------
# work, tolerance, exact results
# ---------------------------------------------------------------------------
def _weight_bytes(n: int, k: int, bits: int, group: int) -> float:
    return n * k * bits / 8 + n * -(-k // group) * 8


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "layer":
        m, h, i, q = case["m"], case["hidden"], case["inter"], case["qkv"]
        nbytes = flops = 0.0
        for n, k in ((q, h), (h, h), (2 * i, h), (h, i)):
            nbytes += _weight_bytes(n, k, case["bits"], case["group"]) + 2.0 * m * n
            flops += 2.0 * m * n * k
        nbytes += 2.0 * m * (h + i)
        return {"bytes": nbytes * case["layers"], "flops": flops * case["layers"]}
    if kind in ("head", "verify"):
        m = case["m"] if kind == "head" else case["c"] * (case["depth"] + 1)
        n, k = case["vocab"], case["hidden"]
        return {"bytes": _weight_bytes(n, k, case["bits"], case["group"]) + 2.0 * m * (n + k),
                "flops": 2.0 * m * n * k}
    if kind == "accept":
        rows = case["c"] * (case["depth"] + 1)
        return {"bytes": 2.0 * rows * case["vocab"] + rows * 20 * 10 + case["c"] * case["depth"] * 260,
                "flops": 0}
    if kind == "greedy":
        return {"bytes": 2.0 * case["rows"] * case["vocab"] + 9 * case["rows"], "flops": 0}
    if kind == "moe":
        t, h, i, e, top_k = case["tokens"], case["hidden"], case["inter"], case["experts"], case["top_k"]
        routes = t * top_k
        # experts that some token is expected to choose: the others are not read
        used = e * (1.0 - (1.0 - top_k / e) ** t)
        weights = (_weight_bytes(2 * i, h, case["bits"], case["group"])
                   + _weight_bytes(h, i, case["bits"], case["group"]))
        nbytes = used * weights + 2.0 * t * (e + h) + 2.0 * routes * (3 * i + h) + 12.0 * routes
        return {"bytes": nbytes, "flops": 6.0 * routes * h * i}
    n, h, bits, t = case["vocab"], case["hidden"], case["bits"], case["tokens"]
    return {"bytes": t * (_weight_bytes(1, h, bits, case["group"]) + 2.0 * h + 8), "flops": 0}


def tolerance(case: dict):
    if case["kind"] in ("accept", "greedy", "embed"):
        return "exact"
    # 16-bit outputs of 32-bit sums, against the same contraction in 64 bits:
    # one rounding to bf16 (measured 1.7e-3) or fp16 (2.1e-4)
    if case.get("dtype") == "fp16":
        return {"rel": 9e-4, "max": 5e-3}
    return {"rel": 7e-3, "max": 4e-2}


def _decode(w: qz.QuantizedMatrix, dtype, rows=slice(None)) -> torch.Tensor:
    """The format's weights (32-bit, one operation after another) rounded to
    ``dtype``, in 64 bits."""
    n, k = w.shape
    bits, group, p = w.encoding.bits, w.encoding.group_in, w.payload
    packed = p["weight_packed"][rows]
    count, dev = packed.shape[0], packed.device
    words = torch.zeros((count, k // 8, 8), dtype=torch.uint8, device=dev)
    words[:, :, :bits] = packed.view(count, k // 8, bits)
    words = words.view(torch.int64)
    shifts = torch.arange(8, device=dev, dtype=torch.int64) * bits
    raw = ((words >> shifts) & ((1 << bits) - 1)).reshape(count, k)
    spread = lambda t: t[rows].float().repeat_interleave(group, dim=1)[:, :k]
    s = spread(p["weight_scale"])
    if bits == 1:
        return ((raw * 2 - 1).float() * s).to(dtype).double()
    q = torch.where(raw >= 1 << (bits - 1), raw - (1 << bits), raw)
    del raw, words
    a, b = spread(p["weight_a"]), spread(p["weight_b"])
    t = (q.abs().double() / ((1 << (bits - 1)) - 1)).float()
    value = t * ((1.0 - a) - b)
    value = t * (b + value)
    value = t * (a + value)
    value = s * value
    return torch.where(q < 0, -value, value).to(dtype).double()


def _product(x: torch.Tensor, w: qz.QuantizedMatrix) -> torch.Tensor:
    """x . decode(w)^T in 64 bits, by slices of w's rows."""
    n, k = w.shape
    x64, step = x.double(), max(1, (1 << 25) // k)
    return torch.cat([x64 @ _decode(w, x.dtype, slice(r, min(n, r + step))).t().contiguous()
                      for r in range(0, n, step)], dim=1)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "layer":
        outputs = []
        for x, x_down, (qkv, o, gate, up, down) in _layer_inputs(case, _generator(seed)):
            outputs += [_product(x, w) for w in (qkv, o, gate, up)] + [_product(x_down, down)]
        return outputs
    if kind == "head":
        gen = _generator(seed)
        x = _normal(gen, (case["m"], case["hidden"]), DTYPES[case["dtype"]])
        return [_product(x, _payload(gen, case["vocab"], case["hidden"], case["bits"], case["group"]))]
    if kind == "verify":
        _, weight, x, _ = _verify_inputs(case, seed)
        return [_product(x, weight), None, None, None]
    if kind == "accept":
        _, target, *_ = _accept_inputs(case, seed)
        scores, ids = torch.sort(target.double(), dim=-1, descending=True, stable=True)
        return [scores[:, :20].contiguous(), ids[:, :20].contiguous(), None, None, None]
    if kind == "greedy":
        return [_greedy_logits(case, seed).double().argmax(-1),
                torch.ones((), dtype=torch.bool, device=_device())]
    if kind == "moe":
        router, x, x_down, (gate, up, down) = _moe_inputs(case, seed)
        e, top_k, inter = case["experts"], case["top_k"], case["inter"]
        order = torch.sort(router.double(), dim=-1, descending=True, stable=True).indices[:, :top_k]
        ids = torch.sort(order, dim=-1).values
        weights = torch.softmax(torch.gather(router.double(), 1, ids), dim=-1)
        h = torch.empty((x_down.shape[0], 2 * inter), dtype=torch.float64, device=x.device)
        y = torch.empty((x_down.shape[0], case["hidden"]), dtype=torch.float64, device=x.device)
        flat = ids.reshape(-1)
        for j in range(e):
            routes = (flat == j).nonzero()[:, 0]
            if routes.numel():
                part = lambda w: w.rows(j * (w.shape[0] // e), (j + 1) * (w.shape[0] // e))
                rows = x[routes // top_k]
                h[routes, :inter] = _product(rows, part(gate))
                h[routes, inter:] = _product(rows, part(up))
                y[routes] = _product(x_down[routes], part(down))
        return [ids, weights, h, y]
    table, ids = _embed_inputs(case, seed)
    dtype = DTYPES[case["dtype"]]
    return [torch.cat([_decode(table, dtype, part) for part in ids.split(1024)])]
