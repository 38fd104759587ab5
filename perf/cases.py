"""Timed cases of the HERM hot path on one GPU, through the package's public fronts.

Families (``op``):

* ``prefill``: a prompt through the whole block stack (``herm.SequencePrefill``);
* ``decode``: one position through the stack at a serving batch (``herm.DecodeGraph``),
  the ids chosen by the caller;
* ``block``: one HERM block over a padded prompt with the state carried in
  (``herm.block_sequence``);
* ``moe``: route, permute, expert GLU FFN and combine (``moe``);
* ``scan``: the affine state scan (``dense.dense_affine_scan``), alone or with its backward;
* ``norm``: RMSNorm-SiLU (``core.fused_rmsnorm_silu``), alone or with its backward;
* ``surprise``: causal surprise with its backward (``think.causal_surprise``);
* ``admission``: surprise from logits and the quantile admission (``think``);
* ``gates``: the recurrent gates and the working-state scan in fp32 (``recurrent.recurrent_scan``).

``listed`` names the sizes of the package's own configurations and of its
operator benchmarks plus one ragged size where a path has one; ``draw`` gives
further sizes, data types and options of the same families. ``exact`` restates
each family in float64 with plain torch.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
from torch.nn import functional

_PACKAGE = Path(__file__).resolve().parent.parent / "koemi-5hom_amd"
if str(_PACKAGE) not in sys.path:
    sys.path.insert(0, str(_PACKAGE))

from koemi_amd import core, dense, herm, moe, recurrent, think  # noqa: E402

PAD = 256
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}
SIZE = {"fp32": 4, "bf16": 2, "fp16": 2}


def listed():
    return [
        # a batch of prompts before generation: the whole 12-layer stack, the package's headline
        {"name": "prefill_8x2048", "op": "prefill", "layers": 12, "width": 1024, "experts": 16, "batch": 8, "length": 2048},
        # one generated position at the serving batch, next ids chosen by the caller
        {"name": "decode_b64", "op": "decode", "layers": 12, "width": 1024, "experts": 16, "batch": 64},
        # one block over ragged prompts padded to a common length, refine memory on, state carried in
        {"name": "block_refine_8x1024", "op": "block", "width": 1024, "experts": 16, "batch": 8, "length": 1024,
         "refine": True, "padded": True},
        # the expert layer of a large token batch with the learned gate (inputs already checked)
        {"name": "moe_32768_bf16", "op": "moe", "tokens": 32768, "width": 1024, "hidden": 2816, "experts": 16, "top_k": 2,
         "dtype": "bf16", "routing": "learned", "padded": False, "validate": False},
        # a ragged batch in half precision, sizes off the tiles, hash routing, padding, the fronts' checks on
        {"name": "moe_3000_fp16", "op": "moe", "tokens": 3000, "width": 768, "hidden": 2000, "experts": 12, "top_k": 2,
         "dtype": "fp16", "routing": "hash", "padded": True, "validate": True},
        # state update of a long prefill
        {"name": "scan_32x4096x1024", "op": "scan", "batch": 32, "length": 4096, "features": 1024, "dtype": "fp32",
         "broadcast": False, "train": False},
        # state update in a training step at the small configuration, with its gradients
        {"name": "scan_train_4x1024x256", "op": "scan", "batch": 4, "length": 1024, "features": 256, "dtype": "fp32",
         "broadcast": False, "train": True},
        # the norm of a training batch, with its gradients
        {"name": "norm_train_32768x512", "op": "norm", "rows": 32768, "hidden": 512, "dtype": "bf16", "train": True},
        # the smallest call: the norm of a few rows in inference, where latency counts
        {"name": "norm_32x512", "op": "norm", "rows": 32, "hidden": 512, "dtype": "fp32", "train": False},
        # the surprise head of a training batch, with its gradients
        {"name": "surprise_train_16x2048x512", "op": "surprise", "batch": 16, "length": 2048, "width": 512, "vocab": 256,
         "dtype": "bf16", "padded": True},
        # scoring a prefill's logits and admitting its most surprising tenth
        {"name": "admission_32768x256", "op": "admission", "rows": 32768, "vocab": 256, "padded": False},
        # gates and working states of a prompt in full precision
        {"name": "gates_8x2048x1024", "op": "gates", "batch": 8, "length": 2048, "width": 1024, "padded": True},
    ]


def _log(rng, low, high):
    """An integer spread over the logarithm of [low, high]."""

    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    op = rng.choice(("prefill", "decode", "block", "moe", "moe", "scan", "scan", "norm", "norm", "surprise", "surprise",
                     "admission", "gates"))
    padded = rng.random() < 0.5
    if op == "prefill":
        return {"op": op, "layers": rng.randint(2, 12), "width": 1024, "experts": 16, "batch": rng.randint(1, 8),
                "length": 128 * _log(rng, 1, 16)}
    if op == "decode":
        return {"op": op, "layers": rng.randint(2, 12), "width": rng.choice((512, 1024)), "experts": rng.choice((8, 16)),
                "batch": _log(rng, 1, 64)}
    if op == "block":
        return {"op": op, "width": rng.choice((256, 512, 1024)), "experts": rng.choice((8, 16)), "batch": rng.randint(1, 8),
                "length": 128 * _log(rng, 1, 16), "refine": rng.random() < 0.5, "padded": padded}
    if op == "moe":
        dtype = rng.choice(("bf16", "bf16", "bf16", "fp16", "fp32"))
        case = {"op": op, "tokens": _log(rng, 1, 32768 if dtype == "bf16" else 6000),
                "width": rng.choice((256, 512, 768, 1000, 1024)), "hidden": rng.choice((512, 1024, 1400, 2048, 2816)),
                "experts": rng.randint(4, 32), "top_k": rng.randint(1, 3), "dtype": dtype,
                "routing": rng.choice(("learned", "hash")), "padded": padded, "validate": rng.random() < 0.5}
        if case["routing"] == "hash":
            case["top_k"] = min(case["top_k"], 2)
        return case
    if op == "scan":
        batch, length, features = _log(rng, 1, 32), _log(rng, 64, 4096), _log(rng, 64, 1024)
        return {"op": op, "batch": batch, "length": length, "features": features,
                "dtype": rng.choice(("fp32", "fp32", "bf16", "fp16")), "broadcast": rng.random() < 0.2,
                "train": rng.random() < 0.6}
    if op == "norm":
        hidden = rng.choice((_log(rng, 64, 4096), 64 * rng.randint(1, 32)))
        return {"op": op, "rows": _log(rng, 16, 1 << min(17, 27 - hidden.bit_length())), "hidden": hidden,
                "dtype": rng.choice(("fp32", "bf16", "bf16", "fp16")), "train": rng.random() < 0.6}
    if op == "surprise":
        return {"op": op, "batch": rng.randint(1, 16), "length": _log(rng, 16, 2048), "width": rng.choice((128, 300, 512, 1024)),
                "vocab": rng.choice((256, 256, 256, 1000)), "dtype": rng.choice(("fp32", "bf16", "bf16", "fp16")),
                "padded": padded}
    if op == "admission":
        return {"op": op, "rows": _log(rng, 64, 65536), "vocab": rng.choice((256, 256, 1000)), "padded": padded}
    return {"op": "gates", "batch": rng.randint(1, 8), "length": _log(rng, 16, 2048), "width": rng.choice((128, 256, 512, 1024)),
            "padded": padded}


# ------------------------------------------------------------------ inputs


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape, scale=1.0, dtype=torch.float32):
    return (torch.randn(shape, generator=g, device="cuda") * scale).to(dtype)


def _uniform(g, *shape, low=0.0, high=1.0, dtype=torch.float32):
    return (torch.rand(shape, generator=g, device="cuda") * (high - low) + low).to(dtype)


def _ids(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.int64)


def _lengths(g, case, batch, length):
    """[B, L] validity: rows of different lengths when padded, else all valid."""

    if not case["padded"]:
        return torch.ones((batch, length), dtype=torch.bool, device="cuda")
    ends = torch.randint((length + 1) // 2, length + 1, (batch, 1), generator=g, device="cuda")
    return torch.arange(length, device="cuda")[None] < ends


def _linear_init(g, *shape):
    """nn.Linear's default initialisation, in values that bf16 holds (a half-precision checkpoint)."""

    bound = 1.0 / math.sqrt(shape[-1])
    bias = shape[:-1]
    return (_uniform(g, *shape, low=-bound, high=bound).bfloat16().float(),
            _uniform(g, *bias, low=-bound, high=bound).bfloat16().float())


def _settings(case):
    return herm.HermSettings(width=case["width"], expert_count=case["experts"], layers=case.get("layers", 1),
                             ablation="herm" if case.get("refine") else "no_refine")


def _weights(g, case, head_scale):
    """Every layer's parameters under the reference modules' names."""

    d, e, m = case["width"], case["experts"], 16
    layers = []
    for layer in range(case.get("layers", 1)):
        p = {}
        if layer == 0:
            p["embedding"] = _randn(g, PAD + 1, d)
            p["embedding"][PAD] = 0.0
        for name in ("input_norm", "fusion_norm", "expert_norm"):
            p[name] = 1.0 + _randn(g, d, scale=0.02)
        for name in ("retention", "candidate", "key", "query", "value", "local_key", "local_value"):
            p[name + "_w"], p[name + "_b"] = _linear_init(g, d, d)
        p["feature_w"], p["feature_b"] = _linear_init(g, m, d)
        p["decay_w"], p["decay_b"] = _linear_init(g, 1, d)
        p["write_w"], p["write_b"] = _linear_init(g, 1, d)
        p["fusion_w"], p["fusion_b"] = _linear_init(g, d, 4 * d)
        for name, shape in (("gate", (e, 2 * d, d)), ("up", (e, 2 * d, d)), ("down", (e, d, 2 * d))):
            p[name + "_w"], p[name + "_b"] = _linear_init(g, *shape)
        head, bias = _linear_init(g, PAD + 1, d)
        p["head_w"], p["head_b"] = head * head_scale, bias * head_scale
        if case.get("refine"):
            p["refine_gate_w"], p["refine_gate_b"] = _linear_init(g, 1, 4 * d)
        layers.append(p)
    return layers


def _carried(g, case):
    """A state in the middle of a conversation: rings mostly full, invalid slots zero."""

    d, b, m, ring = case["width"], case["batch"], 16, 16
    last = _ids(g, b)
    states = []
    for _ in range(case.get("layers", 1)):
        state = {"working": _randn(g, b, d, scale=0.3), "basis": _randn(g, b, d, m, scale=0.1),
                 "normalizer": _uniform(g, b, m, low=0.1, high=1.0), "last_token": last}
        if case.get("refine"):
            state["refine_basis"] = _randn(g, b, d, m, scale=0.05)
            state["refine_normalizer"] = _uniform(g, b, m, low=0.1, high=1.0)
        for name in ("local", "salient"):
            valid = _uniform(g, b, ring) < 0.8
            state[name + "_keys"] = _randn(g, b, ring, d, scale=0.3) * valid[..., None]
            state[name + "_values"] = _randn(g, b, ring, d, scale=0.3) * valid[..., None]
            state[name + "_valid"] = valid
        states.append(state)
    return states


def _inputs(case, seed):
    """The case's tensors, made from the seed alone."""

    g = _generator(seed)
    op = case["op"]
    if op in ("prefill", "decode", "block"):
        # the block's head is scaled so that a good part of its tokens is admitted to the salient memory
        weights = _weights(g, case, 8.0 if op == "block" else 1.0)
        if op == "prefill":
            ids = _ids(g, case["batch"], case["length"])
            return {"weights": weights, "ids": ids, "states": herm.initial_states(_settings(case), case["batch"], ids.device)}
        if op == "decode":
            return {"weights": weights, "ids": _ids(g, 8, case["batch"], 1), "states": _carried(g, case)}
        valid = _lengths(g, case, case["batch"], case["length"])
        ids = torch.where(valid, _ids(g, case["batch"], case["length"]), PAD)
        return {"weights": weights, "ids": ids, "states": _carried(g, case)}
    if op == "moe":
        t, d, h, e, dtype = case["tokens"], case["width"], case["hidden"], case["experts"], DTYPES[case["dtype"]]
        s = {"context": _randn(g, t, d, dtype=dtype),
             "valid": _uniform(g, t) < 0.9 if case["padded"] else torch.ones(t, dtype=torch.bool, device="cuda")}
        for name, shape in (("gate", (e, h, d)), ("value", (e, h, d)), ("output", (e, d, h))):
            s[name + "_w"] = _randn(g, *shape, scale=0.02, dtype=dtype)
            s[name + "_b"] = _randn(g, *shape[:2], scale=0.02, dtype=dtype)
        if case["routing"] == "learned":
            s["router_logits"] = _randn(g, t, e)
        else:
            s["ids"] = _ids(g, t)
            s["previous"] = torch.cat((s["ids"].new_full((1,), PAD), s["ids"][:-1]))
        return s
    if op == "scan":
        b, l, f, dtype = case["batch"], case["length"], case["features"], DTYPES[case["dtype"]]
        s = {"a": torch.sigmoid(_randn(g, b, l, 1 if case["broadcast"] else f) + 2.0).to(dtype),
             "b": _randn(g, b, l, f, scale=0.5, dtype=dtype), "h0": _randn(g, b, f, scale=0.3, dtype=dtype)}
        if case["train"]:
            s["grad"] = _randn(g, b, l, f, dtype=dtype)
        return s
    if op == "norm":
        r, h, dtype = case["rows"], case["hidden"], DTYPES[case["dtype"]]
        s = {"x": _randn(g, r, h, dtype=dtype), "w": (1.0 + _randn(g, h, scale=0.02)).to(dtype)}
        if case["train"]:
            s["grad"] = _randn(g, r, h, dtype=dtype)
        return s
    if op == "surprise":
        b, l, d, v, dtype = case["batch"], case["length"], case["width"], case["vocab"], DTYPES[case["dtype"]]
        return {"prior": _randn(g, b, l, d, scale=0.5, dtype=dtype), "w": _randn(g, v, d, scale=2.0 / math.sqrt(d), dtype=dtype),
                "bias": _randn(g, v, scale=0.1, dtype=dtype), "targets": torch.randint(0, v, (b, l), generator=g, device="cuda"),
                "valid": _lengths(g, case, b, l), "grad": _randn(g, b, l, dtype=dtype)}
    if op == "admission":
        r, v = case["rows"], case["vocab"]
        return {"logits": _randn(g, r, v, scale=2.0), "targets": torch.randint(0, v, (r,), generator=g, device="cuda"),
                "valid": _uniform(g, r) < 0.9 if case["padded"] else torch.ones(r, dtype=torch.bool, device="cuda")}
    b, l, d = case["batch"], case["length"], case["width"]
    s = {"u": _randn(g, b, l, d), "valid": _lengths(g, case, b, l), "h0": _randn(g, b, d, scale=0.3)}
    for name in ("r", "c"):
        bound = 1.0 / math.sqrt(d)
        s["w" + name] = _uniform(g, d, d, low=-bound, high=bound)
        s["b" + name] = _uniform(g, d, low=-bound, high=bound)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    op = case["op"]
    if op in ("prefill", "decode", "block"):
        settings = _settings(case)
        s["settings"] = settings
        s["params"] = herm.prepare_stack(s.pop("weights"), settings, torch.device("cuda"))
        if op == "prefill":
            s["graph"] = herm.SequencePrefill(s["params"], settings, s["states"], s["ids"])
        elif op == "decode":
            s["graph"], s["step"] = herm.DecodeGraph(s["params"], settings, s["ids"][0], s["states"]), 0
    elif op in ("scan", "surprise") or (op == "norm" and case["train"]):
        for name in ("a", "b", "h0", "x", "w", "prior", "bias"):
            if name in s and case.get("train", True):
                s[name].requires_grad_(True)
    s["case"] = case
    return s


# ------------------------------------------------------------------ one pass


def _kept(state):
    """A block's carried state without the salient ring and the token bookkeeping (an entry whose
    score lies within rounding of the threshold moves every later slot of that ring)."""

    return {k: v for k, v in state.items() if not k.startswith("salient") and k not in ("last_token", "local_valid")}


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "prefill":
        graph = s["graph"]
        return {"logits": graph.run(), "surprise": graph.surprise, "state": _kept(graph.states[-1])}
    if op == "decode":
        graph = s["graph"]
        graph.ids.copy_(s["ids"][s["step"] % 8])
        s["step"] += 1
        return {"logits": graph.run(), "state": _kept(graph.states[-1])}
    if op == "block":
        logits, context, state, surprise = herm.block_sequence(s["params"][0], s["settings"], s["ids"], s["states"][0])
        return {"logits": logits, "context": context, "surprise": surprise, "state": _kept(state)}
    if op == "moe":
        return _run_moe(s, case)
    if op == "scan":
        states = dense.dense_affine_scan(s["a"], s["b"], s["h0"])
        if not case["train"]:
            return states
        return (states, *torch.autograd.grad(states, (s["a"], s["b"], s["h0"]), s["grad"]))
    if op == "norm":
        y = core.fused_rmsnorm_silu(s["x"], s["w"])
        return (y, *torch.autograd.grad(y, (s["x"], s["w"]), s["grad"])) if case["train"] else y
    if op == "surprise":
        score = think.causal_surprise(s["prior"], s["w"], s["bias"], s["targets"], s["valid"], validate_targets=False)
        return (score, *torch.autograd.grad(score, (s["prior"], s["w"], s["bias"]), s["grad"]))
    if op == "admission":
        score = think.surprise_from_logits(s["logits"], s["targets"], s["valid"])
        mask, tau = think.salience_admission(score, s["valid"], quantile=0.9)
        return {"score": score, "mask": mask, "tau": tau}
    return recurrent.recurrent_scan(s["u"], s["wr"], s["br"], s["wc"], s["bc"], s["valid"], s["h0"])


def _run_moe(s, case):
    k, e, check = case["top_k"], case["experts"], {"validate": case["validate"]}
    weights = None
    if case["routing"] == "learned":
        assignments, weights = moe.route_topk_learned(s["router_logits"], s["valid"], top_k=k)
    else:
        assignments = moe.route_topk_valid(s["ids"], s["previous"], s["valid"], expert_count=e, top_k=k, **check)
    context, rows, experts, offsets, *pair = moe.permute_topk(s["context"], assignments, s["valid"], expert_count=e,
                                                              pair_weights=weights, **check)
    out = moe.grouped_expert_mlp_inference(context, experts, offsets, s["gate_w"], s["gate_b"], s["value_w"], s["value_b"],
                                           s["output_w"], s["output_b"], **check)
    y = moe.combine_topk(out, rows, offsets, token_count=case["tokens"], top_k=k, pair_weights=pair[0] if pair else None, **check)
    return {"y": y, "assignments": assignments, "offsets": offsets}


# ------------------------------------------------------------------ what a pass cannot do without


def _block_work(case, tokens, window):
    """Bytes and operations of one block over ``tokens`` positions: weights and states once, the
    context in and out; the projections, the content head, two experts a token, the reads."""

    d, e = case["width"], case["experts"]
    weights = 2 * (2 * d * d + (3 * d + 34) * d + 4 * d * d + PAD * d + e * 6 * d * d)
    per_state = case["batch"] * 4 * (d + 16 * d + 16 + 64 * d) * 2
    flops = 2 * d * (2 * d + 3 * d + 34 + 4 * d + PAD) + 2 * 12 * d * d + 4 * d * (16 + 16 + 16 + window // 2)
    if case.get("refine"):
        flops += 4 * d * (16 + window // 2)
    return weights + per_state + tokens * 8 * d, tokens * flops


def work(case):
    op = case["op"]
    if op in ("prefill", "decode", "block"):
        tokens, window = case["batch"] * case.get("length", 1), min(128, case.get("length", 1))
        nbytes, flops = _block_work(case, tokens, window)
        layers, head = case.get("layers", 1), tokens * (PAD + 1)
        return {"bytes": layers * nbytes + 4 * head, "flops": layers * flops + 2 * case["width"] * head}
    if op == "moe":
        t, d, h, e, size = case["tokens"], case["width"], case["hidden"], case["experts"], SIZE[case["dtype"]]
        pairs = t * case["top_k"]
        return {"bytes": size * (min(e, pairs) * 3 * d * h + 2 * t * d) + 16 * pairs, "flops": 6 * d * h * pairs}
    if op == "scan":
        b, l, f, size = case["batch"], case["length"], case["features"], SIZE[case["dtype"]]
        a, x = b * l * (1 if case["broadcast"] else f), b * l * f
        return {"bytes": size * (2 * a + 3 * x + x if case["train"] else a + 2 * x), "flops": (8 if case["train"] else 2) * x}
    if op == "norm":
        x, size = case["rows"] * case["hidden"], SIZE[case["dtype"]]
        return {"bytes": size * x * (4 if case["train"] else 2), "flops": x * (24 if case["train"] else 8)}
    if op == "surprise":
        rows, d, v, size = case["batch"] * case["length"], case["width"], case["vocab"], SIZE[case["dtype"]]
        return {"bytes": size * (2 * rows * d + 2 * v * d + 2 * rows) + 9 * rows, "flops": 6 * rows * d * v}
    if op == "admission":
        return {"bytes": case["rows"] * (4 * case["vocab"] + 8 + 1 + 4 + 1), "flops": case["rows"] * 4 * case["vocab"]}
    rows, d = case["batch"] * case["length"], case["width"]
    return {"bytes": 4 * (2 * rows * d + 2 * d * d), "flops": 4 * rows * d * d}


def tolerance(case):
    """About four times the distance measured from the float64 restatement: 6e-3 for the stack's
    logits, 8e-3 for a block whose admissions may flip, 3e-3 (bf16) and 3e-4 (fp16) for the experts,
    1.7e-3 and 2.2e-4 for one rounding of a result, below 1e-6 for fp32."""

    op = case["op"]
    if op in ("prefill", "decode", "block"):
        return {"rel": {"prefill": 2.4e-2, "decode": 2e-2, "block": 3e-2}[op]}
    if op == "moe":
        return {"rel": {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 1e-5}[case["dtype"]]}
    if op in ("scan", "norm", "surprise"):
        return {"rel": {"bf16": 7e-3, "fp16": 9e-4, "fp32": 1e-5}[case["dtype"]]}
    if op == "admission":
        return {"rel": 1e-5, "differ": 1e-4}
    return {"rel": 1e-5}


# ------------------------------------------------------------------ the same in 64 bits


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w


def _scan64(a, b, h):
    out = torch.empty_like(b)
    for t in range(b.shape[1]):
        h = a[:, t] * h + b[:, t]
        out[:, t] = h
    return out


def _read64(keys, values, eligible, queries):
    """Masked attention read; a query with no eligible slot reads zeros."""

    scores = queries @ keys.transpose(1, 2).contiguous() / math.sqrt(queries.shape[-1])
    scores = scores.masked_fill(~eligible, -math.inf)
    some = eligible.any(-1, keepdim=True)
    return torch.softmax(scores.masked_fill(~some, 0.0), -1).where(some, scores.new_zeros(())) @ values


def _memory64(basis, normalizer, decay, value, features, weight, query):
    """The associative memory's reads before each write, and its final state."""

    log = torch.log(decay)
    total = log.cumsum(1)
    prior = total - log
    length = decay.shape[1]
    past = torch.ones((length, length), dtype=torch.bool, device=decay.device).tril(-1)
    pair = torch.where(past, torch.exp((prior[:, :, None] - total[:, None]).masked_fill(~past, 0.0)), 0.0)
    influence = pair * (query @ features.transpose(1, 2)) * weight[:, None]
    start = torch.exp(prior)
    numerator = start[..., None] * (query @ basis.transpose(1, 2)) + influence @ value
    denominator = (start * (query @ normalizer[..., None])[..., 0] + influence.sum(-1))[..., None]
    floor = denominator + 2.0**-8
    last = torch.exp(total[:, -1:] - total) * weight
    end = torch.exp(total[:, -1])
    return ((denominator / floor) * numerator / floor,
            end[:, None, None] * basis + (value * last[..., None]).transpose(1, 2) @ features,
            end[:, None] * normalizer + (last[:, None] @ features)[:, 0])


def _hash64(ids, previous, experts, top_k):
    v = (ids * 1000003 + previous * 97409) & 0xFFFFFFFF
    for _ in range(2):
        v = ((v ^ (v >> 16)) * 0x45D9F3B) & 0xFFFFFFFF
    v = v ^ (v >> 16)
    return (v[..., None] + torch.arange(top_k, device=ids.device) * 0x9E3779B9) % experts


def _experts64(x, slots, scale, p, names):
    """Sum over a token's distinct experts of scale x FFN(x); slots < 0: none."""

    out = torch.zeros_like(x)
    for k in range(1, slots.shape[1]):
        repeated = (slots[:, :k] == slots[:, k:k + 1]).any(1)
        slots = slots.clone()
        slots[repeated, k] = -1
    for e in range(p[names[0] + "_w"].shape[0]):
        rows, which = torch.nonzero(slots == e, as_tuple=True)
        if not rows.numel():
            continue
        layer = lambda z, name: z @ p[name + "_w"][e].double().t() + p[name + "_b"][e].double()  # noqa: B023, E731
        u = x[rows]
        y = layer(functional.silu(layer(u, names[0])) * layer(u, names[1]), names[2])
        out.index_add_(0, rows, y * scale[rows, which][:, None])
    return out


def _window64(p, case, s, ids, context):
    """One window through one block: (logits, context, next state, surprise)."""

    lin = lambda x, name: x @ p[name + "_w"].double().t() + p[name + "_b"].double()  # noqa: E731
    f = lambda name: p[name].double()  # noqa: E731
    b, length = ids.shape
    valid = ids != PAD
    keep = valid[..., None]
    u = _rms(f("embedding")[ids] if context is None else context, f("input_norm"))
    a = 2.0**-8 + (1 - 2.0**-7) * torch.sigmoid(lin(u, "retention"))
    inc = (1 - a) * torch.tanh(lin(u, "candidate"))
    ws = _scan64(a.where(keep, a.new_ones(())), inc.where(keep, a.new_zeros(())), s["working"])
    before = torch.cat((s["working"][:, None], ws[:, :-1]), 1)
    content = lin(before, "head")[..., :PAD]
    nll = torch.logsumexp(content, -1) - content.gather(-1, torch.where(valid, ids, 0)[..., None])[..., 0]
    surprise = torch.where(valid, 1 - torch.exp(-nll / math.log(PAD)), 0.0)
    admitted = valid & (surprise > 0.75)
    keys, values = lin(ws, "local_key") * keep, lin(ws, "local_value") * keep
    ring = 16
    every = {k: torch.cat((s["local_" + k], v), 1) for k, v in (("keys", keys), ("values", values), ("valid", valid))}
    at, slot = torch.arange(length, device=ids.device)[:, None] + ring, torch.arange(length + ring, device=ids.device)[None]
    near = ((slot < at) & (slot >= at - ring)) & every["valid"][:, None]
    local = _read64(every["keys"], every["values"], near, ws)
    earlier = torch.ones((length, length), dtype=torch.bool, device=ids.device).tril(-1)
    marked = torch.cat((s["salient_valid"][:, None].expand(b, length, ring), admitted[:, None] & earlier), -1)
    kept = {k: torch.cat((s["salient_" + k], v), 1) for k, v in (("keys", keys), ("values", values), ("valid", admitted))}
    salient = _read64(kept["keys"], kept["values"], marked, ws)

    features = torch.softmax(lin(lin(ws, "key"), "feature"), -1)
    query = torch.softmax(lin(lin(ws, "query"), "feature"), -1)
    value = torch.tanh(lin(ws, "value"))
    decay = 2.0**-12 + (1 - 2.0**-11) * torch.sigmoid(lin(ws, "decay"))[..., 0]
    write = torch.sigmoid(lin(ws, "write"))[..., 0]
    masked = lambda d, w: (d.where(valid, d.new_ones(())), w.where(valid, w.new_zeros(())))  # noqa: E731
    d, w = masked(decay, write * (0.25 + 0.75 * surprise))
    memory, basis, normalizer = _memory64(s["basis"], s["normalizer"], d, value, features, w, query)
    new = {"working": ws[:, -1], "basis": basis, "normalizer": normalizer}
    if case.get("refine"):
        nk, nq = functional.normalize(every["keys"], dim=-1), functional.normalize(ws, dim=-1)
        near_cos = (nq @ nk.transpose(1, 2)).masked_fill(~near, -math.inf).amax(-1)
        novelty = torch.where(near.any(-1), 1 - near_cos, 1.0).clamp(0, 1)
        d, w = masked((1 - (1 - decay) * 0.0625).clamp(max=1 - 2.0**-16), write * surprise * novelty)
        refine, new["refine_basis"], new["refine_normalizer"] = _memory64(
            s["refine_basis"], s["refine_normalizer"], d, (value - memory).clamp(-2, 2), features, w, query)
        memory = memory + torch.sigmoid(lin(torch.cat((ws, memory, refine, local), -1), "refine_gate")) * refine
    fused = _rms(lin(torch.cat((ws, memory, local, salient), -1), "fusion"), f("fusion_norm")).reshape(b * length, -1)

    position = torch.where(valid, torch.arange(1, length + 1, device=ids.device), 0).cummax(1).values
    padded = torch.cat((s["last_token"][:, None], ids), 1)
    previous = padded.gather(1, torch.cat((position.new_zeros((b, 1)), position[:, :-1]), 1))
    slots = torch.where(keep, _hash64(ids, previous, case["experts"], 2), -1).reshape(-1, 2)
    update = _experts64(fused, slots, fused.new_full(slots.shape, 0.5), p, ("gate", "up", "down"))
    final = torch.where(valid.reshape(-1, 1), _rms(fused + update, f("expert_norm")), fused).view(b, length, -1)

    new["last_token"] = padded.gather(1, position[:, -1:])[:, 0]
    for k in every:
        new["local_" + k] = every[k][:, -ring:]
    order = torch.arange(kept["valid"].shape[1], device=ids.device)
    rank = torch.where(kept["valid"], order + order.numel(), order).topk(ring, 1).indices.sort(1).values
    new["salient_valid"] = kept["valid"].gather(1, rank)
    for k in ("keys", "values"):
        new["salient_" + k] = kept[k].gather(1, rank[..., None].expand(-1, -1, ws.shape[-1])) * new["salient_valid"][..., None]
    return lin(final, "head"), final, new, surprise


def _stack64(case, s):
    double = lambda st: {k: v.double() if v.is_floating_point() else v for k, v in st.items()}  # noqa: E731
    ids = s["ids"][0] if case["op"] == "decode" else s["ids"]
    contexts, surprises = None, []
    for layer, p in enumerate(s["weights"]):
        state, parts = double(s["states"][layer]), []
        for at in range(0, ids.shape[1], 128):
            piece = None if contexts is None else contexts[:, at:at + 128]
            logits, context, state, surprise = _window64(p, case, state, ids[:, at:at + 128], piece)
            parts.append((logits, context, surprise))
        logits, contexts, surprise = (torch.cat(x, 1) for x in zip(*parts))
        surprises.append(surprise)
    out = {"logits": logits, "state": _kept(state)}
    if case["op"] == "prefill":
        out["surprise"] = surprises
    if case["op"] == "block":
        out.update(context=contexts, surprise=surprise)
    return out


def exact(case, seed):
    op = case["op"]
    s = _inputs(case, seed)
    if op in ("prefill", "decode", "block"):
        return _stack64(case, s)
    if op == "moe":
        if case["routing"] == "learned":
            scale, slots = torch.topk(torch.softmax(s["router_logits"].double(), -1), case["top_k"], -1)
        else:
            slots = _hash64(s["ids"], s["previous"], case["experts"], case["top_k"])
            scale = torch.full(slots.shape, 1.0 / case["top_k"], dtype=torch.float64, device="cuda")
        slots = torch.where(s["valid"][:, None], slots, -1)
        return {"y": _experts64(s["context"].double(), slots, scale, s, ("gate", "value", "output")), "assignments": None,
                "offsets": None}
    if op == "scan":
        a, b, h = (s[k].double() for k in ("a", "b", "h0"))
        states = _scan64(a, b, h)
        if not case["train"]:
            return states
        before = torch.cat((h[:, None], states[:, :-1]), 1)
        g, carry = s["grad"].double(), torch.zeros_like(h)
        for t in range(b.shape[1] - 1, -1, -1):
            g[:, t] += carry
            carry = a[:, t] * g[:, t]
        da = g * before
        return states, da.sum(-1, keepdim=True) if case["broadcast"] else da, g, carry
    if op == "norm":
        leaves = [s[k].double().requires_grad_(True) for k in ("x", "w")]
        y = functional.silu(_rms(*leaves))
        return (y.detach(), *torch.autograd.grad(y, leaves, s["grad"].double())) if case["train"] else y.detach()
    if op == "surprise":
        leaves = [s[k].double().requires_grad_(True) for k in ("prior", "w", "bias")]
        z = leaves[0] @ leaves[1].t() + leaves[2]
        nll = torch.logsumexp(z, -1) - z.gather(-1, s["targets"][..., None])[..., 0]
        score = torch.where(s["valid"], 1 - torch.exp(-nll / math.log(case["vocab"])), 0.0)
        return (score.detach(), *torch.autograd.grad(score, leaves, s["grad"].double()))
    if op == "admission":
        z = s["logits"].double()
        nll = torch.logsumexp(z, -1) - z.gather(-1, s["targets"][:, None])[:, 0]
        score = torch.where(s["valid"], 1 - torch.exp(-nll / math.log(case["vocab"])), 0.0)
        return {"score": score, "mask": None, "tau": torch.quantile(score, 0.9)}
    u, wr, br, wc, bc, h = (s[k].double() for k in ("u", "wr", "br", "wc", "bc", "h0"))
    keep = s["valid"][..., None]
    a = 2.0**-8 + (1 - 2.0**-7) * torch.sigmoid(u @ wr.t() + br)
    inc = (1 - a) * torch.tanh(u @ wc.t() + bc)
    return _scan64(torch.where(keep, a, 1.0), torch.where(keep, inc, 0.0), h)
