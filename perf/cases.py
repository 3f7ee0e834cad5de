"""The work that users of this framework have it do, as timed cases.

Every case is one pass through the public entry points, on ModernBERT-base
geometry (hidden 768, 12 heads, intermediate 1152, every third layer global,
vocabulary 50368), the one geometry the repository ships:

  serve     single requests answered one after another, host ids in, logits
            out (Engine.forward): an interactive service. Small requests are
            bound by latency and launches, larger ones by how well one
            sequence fills the GPU.
  batch     one forward over many packed requests whose token arrays are on
            the device (Engine.forward_device): a throughput service, offline
            scoring. Several sequence lengths in one batch are the ordinary
            case; equal ones are the benchmark's.
  evaluate  one SystemOne call (dn_evaluate): every question about one state
            in one forward, calibrated probabilities out. It runs in fp16 with
            certified argmax, the mode whose choices are the reference's.
  train     one optimizer step of the trainer: micro-batches within its token
            budget, each forward + loss + backward, then the gradient norm,
            the AdamW update and cleared gradients.
  gemm      one projection product on device operands (Engine.gemm_device,
            gemm_device_store), as a program uses the library's BLAS half.

A training step returns gradients where they are well conditioned and the
updated weights elsewhere: the gradients of the MLP and the norms are sums over
the options' rows that cancel (the loss's derivative sums to zero over a
question's options), so in bf16 they are 5-10% off their float64 values
whatever the order of the sums.

Weights have the statistics of the repository's random models (N(0, 0.02))
with norm weights around 1 and small biases, rounded to bfloat16 as a released
bundle stores them; they do not depend on the seed. Token ids, their packing,
the order of a ragged batch's sequences and the targets come from the seed.
"""
import ctypes
import math

import numpy as np
import torch

from decide_amd.native import check, lib
from decide_amd.nn import MASK_ID, Engine, build_sequence, flatten, modernbert_base, row_tokens, tensor_shapes
from decide_amd.synth import CFG4_ORDER, SEGMENTS, pack_request, random_ids
from decide_amd.train import TrainEngine, soft_cross_entropy

HIDDEN, INTER, HEADS, VOCAB, LAYERS = 768, 1152, 12, 50368, 22
CERTIFY_MARGIN = 1e-3
TEMPERATURE = 1.3
RATE, DECAY = 1e-5, 0.01


def listed():
    return [
        # The smallest question: 40 tokens of premise, two options of 12 (64 tokens). Pure latency.
        {"name": "serve 64 fp16", "kind": "serve", "precision": "fp16", "requests": 16,
         "premise": 40, "options": 2, "option": 12, "spread": 0.0},
        # A page of context with eight options (416 to 608 tokens): the ordinary single request.
        {"name": "serve 512 bf16", "kind": "serve", "precision": "bf16", "requests": 16,
         "premise": 384, "options": 8, "option": 16, "spread": 0.25},
        # A short request in the fp32 mode (validation, and what certification recomputes).
        {"name": "serve 203 fp32", "kind": "serve", "precision": "fp32", "requests": 4,
         "premise": 143, "options": 5, "option": 12, "spread": 0.0},
        # A small dynamic batch: 11 requests of different lengths, about 2,000 tokens, each time in another order.
        {"name": "batch ragged 2k fp16", "kind": "batch", "precision": "fp16", "sequences": 11,
         "premise": 141, "options": 4, "option": 11, "spread": 0.6},
        # The serving shape of the repository's benchmark: 64 requests of 512 tokens.
        {"name": "batch 64x512 bf16", "kind": "batch", "precision": "bf16", "sequences": 64,
         "premise": 384, "options": 8, "option": 16, "spread": 0.0},
        # Long states: 8 requests around 2,800 tokens with 84 options, ragged.
        {"name": "batch long ragged bf16", "kind": "batch", "precision": "bf16", "sequences": 8,
         "premise": 2048, "options": 84, "option": 9, "spread": 0.1},
        # One SystemOne call: 24 questions about a state of about 400 tokens.
        {"name": "evaluate 24 questions", "kind": "evaluate", "questions": 24, "state": 401},
        # The trainer's step: 32 examples of 384 tokens within a token budget of 4,000.
        {"name": "train 32x384 bf16", "kind": "train", "precision": "bf16", "examples": 32,
         "premise": 256, "options": 8, "option": 16, "spread": 0.0, "budget": 4000, "train_from": 0},
        # A fine-tuning step on few ragged examples, the lower layers frozen.
        {"name": "train 6 ragged bf16", "kind": "train", "precision": "bf16", "examples": 6,
         "premise": 113, "options": 3, "option": 13, "spread": 0.5, "budget": 4000, "train_from": 11},
        # The fp32 product of the BLAS benchmark (fused QKV over one request).
        {"name": "gemm 512 fp32", "kind": "gemm", "precision": "fp32", "op": "f32", "m": 512, "n": 2304, "k": 768},
        # The QKV projection of a ragged batch, rounded to bf16 as the forward stores it.
        {"name": "gemm 5003 store bf16", "kind": "gemm", "precision": "bf16", "op": "store", "m": 5003, "n": 2304,
         "k": 768},
        # The MLP output projection added into an fp32 residual at the serving batch.
        {"name": "gemm 32768 add bf16", "kind": "gemm", "precision": "bf16", "op": "add", "m": 32768, "n": 768,
         "k": 1152},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["serve", "serve", "batch", "batch", "evaluate", "train", "gemm"])
    options, option = rng.randint(2, 12), rng.randint(3, 20)
    if kind == "serve":
        precision = rng.choice(["fp16", "bf16", "fp32"])
        premise = _log_int(rng, 17, 300 if precision == "fp32" else 1200)
        return {"kind": kind, "precision": precision, "requests": 4 if precision == "fp32" else 16,
                "premise": premise, "options": options, "option": option, "spread": rng.choice([0.0, 0.4])}
    if kind == "batch":
        precision = rng.choice(["fp16", "bf16"])
        tokens = _log_int(rng, 300, 32000 if precision == "bf16" else 8000)
        per = min(tokens, _log_int(rng, 60, 3000))
        premise = max(17, per - options * option)
        return {"kind": kind, "precision": precision,
                "sequences": max(1, tokens // (premise + options * option)), "premise": premise, "options": options,
                "option": option, "spread": rng.choice([0.0, 0.3, 0.7])}
    if kind == "evaluate":
        return {"kind": kind, "questions": rng.randint(3, 24), "state": _log_int(rng, 60, 440)}
    if kind == "train":
        premise = _log_int(rng, 30, 250)
        return {"kind": kind, "precision": "bf16", "examples": _log_int(rng, 3, 30), "premise": premise,
                "options": rng.randint(2, 8), "option": rng.randint(3, 16), "spread": rng.choice([0.0, 0.5]),
                "budget": rng.choice([2000, 4000]), "train_from": rng.choice([0, 0, 11])}
    precision = rng.choice(["bf16", "bf16", "fp32"])
    n, k = rng.choice([(2304, 768), (768, 768), (768, 1152), (1152, 768), (768, 2304), (1536, 768)])
    return {"kind": kind, "precision": precision, "op": rng.choice(["f32", "add"] if precision == "fp32" else
                                                                   ["store", "f32", "add"]),
            "m": _log_int(rng, 33, 4000 if precision == "fp32" else 32768), "n": n, "k": k}


# ---- the model -------------------------------------------------------------

_CONFIG = modernbert_base()
_WEIGHTS = {}  # tensors of the model by name, float32 on the host
_ENGINES = {}  # the inference engines that a serving program keeps open


def _weights():
    if not _WEIGHTS:
        gen = torch.Generator(device="cuda").manual_seed(20)
        for name, shape in tensor_shapes(_CONFIG).items():
            w = 0.02 * torch.randn(shape, generator=gen, device="cuda")
            if name.endswith("norm.weight"):
                w = 1.0 + 5.0 * w
            _WEIGHTS[name] = w.bfloat16().float().cpu().numpy()
    return _WEIGHTS


def _engine(precision, certify=0.0):
    if (precision, certify) not in _ENGINES:
        _ENGINES[precision, certify] = Engine(_CONFIG, _weights(), precision=precision, certify=certify)
    return _ENGINES[precision, certify]


# ---- inputs ----------------------------------------------------------------

def _premises(case, count):
    """The premise lengths of a batch: `spread` is the relative half width of their range."""
    p, spread = case["premise"], case["spread"]
    return [max(4, int(round(p * (1 + spread * (2 * ((i * 0.6180339887) % 1.0) - 1))))) for i in range(count)]


def _count(case):
    return case.get("sequences") or case.get("requests") or case["examples"]


def _sequences(case, seed):
    rng = np.random.default_rng(seed)
    lens = _premises(case, _count(case))
    return [build_sequence(pack_request(rng, lens[i], [case["option"]] * case["options"], VOCAB), MASK_ID, True)
            for i in rng.permutation(len(lens))]


def _questions(case, seed):
    """(kinds, option counts, ids per question) of one SystemOne call, packed as Local packs it."""
    rng = np.random.default_rng(seed)
    state = random_ids(rng, case["state"], VOCAB)
    code = {"choice": 0, "score": 1, "noul": 2}
    kinds, nopt, ids = [], [], []
    for q in range(case["questions"]):
        kind = CFG4_ORDER[q % len(CFG4_ORDER)]
        parts = [np.array([50281], np.int32), random_ids(rng, 9 + q % 8, VOCAB), state, np.array([50282], np.int32)]
        for n in SEGMENTS[kind]:
            parts += [np.array([MASK_ID], np.int32), random_ids(rng, n - 1, VOCAB)]
        ids.append(np.concatenate(parts + [np.array([50282], np.int32)]).astype(np.int32))
        kinds.append(code[kind])
        nopt.append(len(SEGMENTS[kind]))
    return kinds, nopt, ids


def _micro_batches(case, seed):
    """[(sequences, one-hot targets)] of one step, whole examples within the token budget."""
    seqs = _sequences(case, seed)
    rng = np.random.default_rng(seed + 1)
    out, used = [], case["budget"] + 1
    for s in seqs:
        if used + len(s.ids) > case["budget"]:
            out.append(([], []))
            used = 0
        used += len(s.ids)
        out[-1][0].append(s)
        out[-1][1].append(np.eye(case["options"])[int(rng.integers(0, case["options"]))])
    return out


def _gemm_inputs(case, seed):
    """Activations ~ N(0, 1) and weights ~ N(0, 0.02) in the operand type; the fp32 output or residual."""
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    dtype = torch.float32 if case["precision"] == "fp32" else torch.bfloat16
    a = torch.randn((case["m"], case["k"]), generator=gen, device="cuda").to(dtype)
    b = (0.02 * torch.randn((case["n"], case["k"]), generator=gen, device="cuda")).to(dtype)
    if case["op"] == "store":
        c = torch.empty((case["m"], case["n"]), dtype=dtype, device="cuda")
    elif case["op"] == "add":
        c = torch.randn((case["m"], case["n"]), generator=gen, device="cuda")
    else:
        c = torch.empty((case["m"], case["n"]), device="cuda")
    return a, b, c


def _grad_names(case):
    """The tensors whose gradients a step returns, from the lowest and a middle trainable layer."""
    lo = case["train_from"]
    mid = (lo + LAYERS - 1) // 2
    return ["model.layers.%d.attn.Wqkv.weight" % lo, "model.layers.%d.attn.Wo.weight" % mid]


def _weight_names(case):
    """The tensors that a step returns as updated."""
    lo = case["train_from"]
    mid = (lo + LAYERS - 1) // 2
    return ["model.layers.%d.mlp.Wi.weight" % lo, "model.layers.%d.mlp.Wo.weight" % mid,
            "model.layers.%d.mlp_norm.weight" % lo, "model.layers.%d.attn_norm.weight" % mid, "model.final_norm.weight",
            "scorer.dense.weight", "scorer.out_proj.weight"]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return {"case": case, "engine": _engine(case["precision"]),
                "requests": [[s] for s in _sequences(case, seed)]}
    if kind == "batch":
        seqs = _sequences(case, seed)
        seq_len, ids, pos, opt, _, _ = flatten(seqs)
        rows = row_tokens(seqs)
        put = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        return {"case": case, "engine": _engine(case["precision"]), "seq_len": seq_len,
                "ids": put(ids), "pos": put(pos), "opt": put(opt), "rows": put(rows),
                "logits": torch.zeros(len(rows), dtype=torch.float32, device="cuda")}
    if kind == "evaluate":
        kinds, nopt, ids = _questions(case, seed)
        return {"case": case, "engine": _engine("fp16", CERTIFY_MARGIN),
                "kinds": np.array(kinds, np.int32), "nopt": np.array(nopt, np.int32),
                "len": np.array([len(x) for x in ids], np.int32), "ids": np.concatenate(ids),
                "temperature": np.full(len(ids), TEMPERATURE)}
    if kind == "train":
        engine = TrainEngine(_CONFIG, _weights(), precision=case["precision"], train_from=case["train_from"],
                             train_emb=False)
        return {"case": case, "engine": engine, "micro": _micro_batches(case, seed)}
    a, b, c = _gemm_inputs(case, seed)
    engine = _engine("bf16")
    engine.set_stream(torch.cuda.current_stream().cuda_stream)
    return {"case": case, "engine": engine, "a": a, "b": b, "c": c}


# ---- one pass --------------------------------------------------------------

def _ptr(a):
    return a.ctypes.data_as(ctypes.c_void_p)


def run(state):
    case, engine = state["case"], state["engine"]
    kind = case["kind"]
    if kind == "serve":
        return np.concatenate([engine.forward(request) for request in state["requests"]])
    if kind == "batch":
        engine.forward_device(state["seq_len"], state["ids"].data_ptr(), state["pos"].data_ptr(),
                              state["opt"].data_ptr(), len(state["rows"]), state["rows"].data_ptr(),
                              state["logits"].data_ptr())
        return state["logits"]
    if kind == "evaluate":
        nq, rows = len(state["kinds"]), int(state["nopt"].sum())
        probs, choice = np.zeros(rows), np.zeros(nq, np.int32)
        confidence, value = np.zeros(nq), np.zeros(nq)
        check(lib.dn_evaluate(engine.handle, nq, _ptr(state["kinds"]), _ptr(state["nopt"]), _ptr(state["len"]),
                              _ptr(state["ids"]), _ptr(state["temperature"]), MASK_ID, 1, _ptr(probs), _ptr(choice),
                              _ptr(confidence), _ptr(value)), engine.handle)
        return {"probabilities": probs, "choice": choice, "confidence": confidence, "value": value}
    if kind == "train":
        logits = []
        for seqs, targets in state["micro"]:
            out = engine.forward(seqs)
            _, dlogits = soft_cross_entropy(out, targets, case["examples"])
            engine.backward(dlogits)
            logits.append(out)
        norm = engine.grad_norm()
        grads = {name: engine.download(name, "grad") for name in _grad_names(case)}
        engine.update(RATE, RATE, DECAY, 1.0 if norm <= 1.0 else 1.0 / (norm + 1e-6))
        engine.zero_grad()
        return {"logits": np.concatenate(logits), "norm": norm, "gradients": grads,
                "weights": {name: engine.download(name) for name in _weight_names(case)}}
    a, b, c = state["a"].data_ptr(), state["b"].data_ptr(), state["c"].data_ptr()
    if case["op"] == "store":
        engine.gemm_device_store(case["precision"], case["m"], case["n"], case["k"], a, b, c)
    else:
        engine.gemm_device(case["precision"], case["m"], case["n"], case["k"], a, b, c, case["op"] == "add")
    return state["c"]


# ---- what a pass cannot do without -----------------------------------------

_LAYER = 4 * HIDDEN * HIDDEN + 3 * HIDDEN * INTER  # projection weights of a layer


def _attention_flops(lengths, layers, prefix):
    """Allowed query-key pairs of a few long-or-short sequences, 4 flops per pair and hidden column."""
    total = 0
    for n, p in zip(lengths, prefix):
        full = n * p + (n - p) * (n - p) / 8.0  # every query sees the prefix; options see their own segment
        window = n * min(p, 129)
        globals_ = (layers + 2) // 3
        total += 4 * HIDDEN * (globals_ * full + (layers - globals_) * window)
    return total


def work(case):
    kind = case["kind"]
    if kind == "gemm":
        es = 4 if case["precision"] == "fp32" else 2
        m, n, k = case["m"], case["n"], case["k"]
        out = {"store": es, "f32": 4, "add": 8}[case["op"]]
        return {"bytes": es * (m * k + n * k) + out * m * n, "flops": 2 * m * n * k}
    if kind == "evaluate":
        prefix = [case["state"] + 11 + q % 8 for q in range(case["questions"])]
        lengths, es = [p + 33 for p in prefix], 2
        calls, rows = 1, 4 * case["questions"]
    else:
        prefix = _premises(case, _count(case))
        lengths = [p + case["options"] * case["option"] for p in prefix]
        es = 4 if case["precision"] == "fp32" else 2
        calls, rows = case.get("requests", 1), len(prefix) * case["options"]
    tokens = sum(lengths)
    forward = 2 * tokens * LAYERS * _LAYER + _attention_flops(lengths, LAYERS, prefix)
    weights = es * LAYERS * _LAYER + 4 * (HIDDEN * HIDDEN // 2)
    inputs = tokens * (12 + 4 * HIDDEN) + 8 * rows
    if kind != "train":
        return {"bytes": calls * weights + inputs, "flops": forward}
    trained = LAYERS - case["train_from"]
    # Backward: input and weight gradients of the trainable layers; AdamW reads and writes weights and two moments.
    backward = (2 * tokens * 2 * _LAYER + 2.5 * _attention_flops(lengths, 3, prefix) / 3) * trained
    return {"bytes": weights + inputs + trained * _LAYER * (4 * 7 + 2), "flops": forward + backward}


def tolerance(case):
    """About four times the differences measured: against float64, or for the fp32 products against other orders."""
    kind = case["kind"]
    if kind == "gemm":
        return {"rel": 4e-3 if case["op"] == "store" else 3e-6}
    if kind == "evaluate":
        return {"rel": 6e-3}
    if kind == "train":
        return {"rel": 0.03}
    return {"rel": {"fp32": 5e-6, "fp16": 2e-3, "bf16": 0.02}[case["precision"]]}


# ---- the same in 64 bits ---------------------------------------------------

def _norm64(x, w, eps, b=None):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w, b, eps)


def _rope64(sliding, pos):
    """cos and sin per (token, frequency); the angle is rounded to float32, as the model defines its tables."""
    theta = _CONFIG.local_theta if sliding else _CONFIG.global_theta
    inv = theta ** (-torch.arange(0, 32, dtype=torch.float64, device="cuda") / 32)
    angle = (pos.double()[:, None] * inv).float().double()
    return torch.cos(angle), torch.sin(angle)


def _rotate(x, cs):
    cos, sin = cs
    a, b = x[..., :32], x[..., 32:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _encode64(W, seq):
    """The encoder over one sequence and the scorer over its option rows: float64 logits."""
    put = lambda a: torch.from_numpy(np.asarray(a)).cuda().long()  # noqa: E731
    ids, pos, opt, rows = put(seq.ids), put(seq.pos), put(seq.opt), put(seq.mask_pos)
    n = len(ids)
    sees = (opt[None, :] == -1) | (opt[None, :] == opt[:, None])
    near = sees & ((pos[None, :] - pos[:, None]).abs() <= _CONFIG.half_window)
    rope = {s: _rope64(s, pos) for s in (False, True)}
    gelu = torch.nn.functional.gelu
    h = _norm64(W["model.embeddings.tok_embeddings.weight"][ids], W["model.embeddings.norm.weight"], _CONFIG.eps)
    for i in range(LAYERS):
        p, sliding = "model.layers.%d." % i, _CONFIG.is_sliding(i)
        x = h if i == 0 else _norm64(h, W[p + "attn_norm.weight"], _CONFIG.eps)
        q, k, v = (x @ W[p + "attn.Wqkv.weight"].T).view(n, 3, HEADS, 64).permute(1, 2, 0, 3)
        s = _rotate(q, rope[sliding]) @ _rotate(k, rope[sliding]).transpose(1, 2).contiguous() / 8.0
        s = s.masked_fill(~(near if sliding else sees), -math.inf)
        ctx = (torch.softmax(s, -1) @ v).permute(1, 0, 2).reshape(n, HIDDEN)
        h = h + ctx @ W[p + "attn.Wo.weight"].T
        x = _norm64(h, W[p + "mlp_norm.weight"], _CONFIG.eps) @ W[p + "mlp.Wi.weight"].T
        h = h + (gelu(x[:, :INTER]) * x[:, INTER:]) @ W[p + "mlp.Wo.weight"].T
    x = _norm64(h[rows], W["model.final_norm.weight"], _CONFIG.eps)
    x = _norm64(x, W["scorer.input_norm.weight"], 1e-5, W["scorer.input_norm.bias"])
    x = gelu(x @ W["scorer.dense.weight"].T + W["scorer.dense.bias"])
    x = _norm64(x, W["scorer.norm.weight"], 1e-5, W["scorer.norm.bias"])
    return (x @ W["scorer.out_proj.weight"].T + W["scorer.out_proj.bias"])[:, 0]


def _weights64():
    return {name: torch.from_numpy(w).cuda().double() for name, w in _weights().items()}


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        a, b, c = _gemm_inputs(case, seed)
        out = a.double() @ b.double().T
        return out + c.double() if case["op"] == "add" else out
    if kind == "train":
        W = _weights64()
        for name, w in W.items():
            layer = name.split(".")[2] if name.startswith("model.layers.") else None
            w.requires_grad_(not name.startswith("model.embeddings.") and
                             (layer is None or int(layer) >= case["train_from"]))
        logits = []
        for seqs, targets in _micro_batches(case, seed):
            for seq, target in zip(seqs, targets):
                out = _encode64(W, seq)
                t = torch.from_numpy(np.asarray(target, np.float64)).cuda()
                (-(t * torch.log_softmax(out, 0)).sum() / case["examples"]).backward()
                logits.append(out.detach())
        norm = math.sqrt(sum(float(w.grad.square().sum()) for w in W.values() if w.grad is not None))
        scale = 1.0 if norm <= 1.0 else 1.0 / (norm + 1e-6)
        weights = {}
        for name in _weight_names(case):  # the first AdamW step: both moments' corrections cancel
            w, g = W[name].detach(), scale * W[name].grad
            weights[name] = w - RATE * (g / (g.abs() + 1e-8) + (DECAY * w if w.dim() == 2 else 0.0))
        return {"logits": torch.cat(logits), "norm": norm,
                "gradients": {name: W[name].grad for name in _grad_names(case)}, "weights": weights}
    with torch.no_grad():
        W = _weights64()
        if kind != "evaluate":
            return torch.cat([_encode64(W, seq) for seq in _sequences(case, seed)])
        kinds, _, ids = _questions(case, seed)
        probs, choice, value = [], [], []
        for kind_, row in zip(kinds, ids):
            logits = _encode64(W, build_sequence(row, MASK_ID, True))
            p = torch.softmax(logits / TEMPERATURE, 0)
            probs.append(p)
            choice.append(int(logits.argmax()) if kind_ == 0 else -1)
            value.append(float((p * torch.arange(len(p), device="cuda")).sum()) if kind_ == 1 else
                         float(p[0]) if kind_ == 2 else 0.0)
        return {"probabilities": torch.cat(probs), "choice": np.array(choice, np.int32), "confidence": None,
                "value": np.array(value)}
