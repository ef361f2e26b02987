"""What users of this package have it do, as measurable cases.

A case is a dict of plain values; its "kind" says which entry point it goes through:

  classify   a whole forward: 24 layers and the head (`GLiNERDecideClassifier`), the logits returned
  layer      one encoder layer on the caller's hidden states (`layer_forward`)
  linear     one projection with its epilogue (`FusedKernels.linear`), rows gathered or not
  attention  the closed-form-index attention stage (`FusedKernels.deberta_attention`)
  ln         the residual LayerNorm (`FusedKernels.residual_layer_norm`)
  bias       the relative bias with index tensors (`FusedKernels.relative_bias`)
  fused      the whole attention with index tensors (`FusedKernels.fused_attention`)

Everything is fp16 with fp32 arithmetic, the one data type of the checkpoint.  Widths are the model's
(hidden 1024, 16 heads of 64, intermediate 4096, classifier 2048, 512 relative positions); batch sizes
and lengths range over what the length buckets L32 to L512 and batches of up to 64 rows give.
"""

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PACKAGE = str(Path.cwd() / "gliner-decide-metal_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from gliner_decide import DecisionInput, DeBERTaV2Configuration, FusedKernels, GLiNERDecideClassifier  # noqa: E402
from gliner_decide.synthetic import weight_shapes  # noqa: E402

HIDDEN, HEADS, HEAD_DIM, FFN, POSITIONS, CLS_HIDDEN = 1024, 16, 64, 4096, 512, 2048
LAYERS = 24
EPS = 1e-7
BUCKETS = (32, 64, 96, 128, 256, 512)
LAYER_VOCAB = 2048  # the layer cases never look a token up


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # One short text classified on its own, host arrays in: what an interactive caller waits for.
        # Latency and launches.
        {"name": "classify_one_text_l64", "kind": "classify", "batch": 1, "seq_len": 64, "tasks": 1, "labels": 5,
         "min_len": 40, "host": True},
        # The batch driver's ordinary step and the package's headline: 32 rows of 40 to 256 tokens, packed.
        {"name": "classify_batch_b32_l256", "kind": "classify", "batch": 32, "seq_len": 256, "tasks": 1, "labels": 5,
         "min_len": 40, "host": False},
        # One layer for the smallest bucket, as a caller that runs the encoder layer by layer has it.
        {"name": "layer_b1_l32", "kind": "layer", "batch": 1, "seq_len": 32, "min_len": 32},
        # One layer of the long-context batch, every position computed: the largest case.
        {"name": "layer_b64_l512", "kind": "layer", "batch": 64, "seq_len": 512, "min_len": 512},
        # The QKV projection of the headline batch's packed tokens (not a multiple of any tile).
        {"name": "linear_qkv_m4896", "kind": "linear", "m": 4896, "n": 3072, "k": 1024, "epilogue": "bias",
         "gather_from": 0},
        # The intermediate projection with GELU on a full 32 x 256 batch.
        {"name": "linear_ffn_up_m8192", "kind": "linear", "m": 8192, "n": 4096, "k": 1024, "epilogue": "gelu",
         "gather_from": 0},
        # The output projection of the feed-forward on one or two rows' worth of tokens: a long sum, few rows.
        {"name": "linear_ffn_down_m300", "kind": "linear", "m": 300, "n": 1024, "k": 4096, "epilogue": "bias",
         "gather_from": 0},
        # The classifier's first layer: 5 markers of each of 32 rows gathered from the hidden states, ReLU.
        {"name": "linear_markers_m160", "kind": "linear", "m": 160, "n": 2048, "k": 1024, "epilogue": "relu",
         "gather_from": 8192},
        # Relative bias and masked softmax, probabilities out: the workload that the bias figures are quoted on.
        {"name": "attention_probs_b32_l256", "kind": "attention", "batch": 32, "seq_len": 256, "min_len": 16,
         "output": "probs", "score": "default"},
        # The residual LayerNorm of a full 32 x 256 batch.
        {"name": "residual_ln_8192", "kind": "ln", "rows": 8192, "round_sum": True},
        # The relative bias with the caller's own index tensors, a full batch (every key valid: masked keys are
        # constants of -65504 that would drown every other value of the output in a comparison).
        {"name": "bias_indices_b32_l256", "kind": "bias", "batch": 32, "seq_len": 256, "min_len": 256},
        # Attention with the caller's own index tensors on rows that were not padded to a bucket.
        {"name": "fused_indices_b8_l200", "kind": "fused", "batch": 8, "seq_len": 200, "min_len": 16},
    ]


def _log(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("classify", "layer", "linear", "linear", "attention", "ln", "bias", "fused"))
    if kind == "classify":
        seq_len = rng.choice(BUCKETS)
        tasks = rng.randint(1, 2)
        labels = rng.randint(2, 10) if seq_len > 32 else rng.randint(2, 5)
        min_len = rng.randint(2 + tasks * labels, seq_len)
        batch = _log(rng, 1, min(32, 2 * 4400 // (min_len + seq_len)))
        return {"kind": kind, "batch": batch, "seq_len": seq_len, "tasks": tasks, "labels": labels,
                "min_len": min_len, "host": batch == 1}
    if kind == "layer":
        seq_len = 16 * rng.randint(1, 32)
        return {"kind": kind, "batch": _log(rng, 1, min(64, 32768 // seq_len)), "seq_len": seq_len,
                "min_len": rng.randint(1, seq_len)}
    if kind == "linear":
        n, k, epilogue = rng.choice(((3072, 1024, "bias"), (1024, 1024, "bias"), (4096, 1024, "gelu"),
                                     (1024, 4096, "bias"), (2048, 1024, "relu")))
        if epilogue == "relu":  # marker rows: batch x tasks x labels of them
            rows = _log(rng, 32, 16384)
            return {"kind": kind, "m": min(rows, _log(rng, 2, 4096)), "n": n, "k": k, "epilogue": epilogue,
                    "gather_from": rows}
        return {"kind": kind, "m": _log(rng, 16, 16384), "n": n, "k": k, "epilogue": epilogue, "gather_from": 0}
    if kind == "attention":
        seq_len = 16 * rng.randint(1, 32)
        return {"kind": kind, "batch": _log(rng, 1, min(64, 32 * 256 * 256 // (seq_len * seq_len))),
                "seq_len": seq_len, "min_len": rng.randint(1, seq_len), "output": rng.choice(("probs", "context")),
                "score": rng.choice(("default", "default", "explicit", "kernel_bias", "fused"))}
    if kind == "ln":
        return {"kind": kind, "rows": _log(rng, 16, 32768), "round_sum": rng.random() < 0.5}
    seq_len = _log(rng, 16, 512)  # any length, not only multiples of a tile
    return {"kind": kind, "batch": _log(rng, 1, max(1, min(32, 8 * 512 * 512 // (seq_len * seq_len)))),
            "seq_len": seq_len, "min_len": seq_len if kind == "bias" else rng.randint(1, seq_len)}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    return (x * std + mean).to(torch.float16)


def _lengths(seed, case):
    r = np.random.default_rng([int(seed), 77])
    return r.integers(case["min_len"], case["seq_len"] + 1, size=case["batch"])


def _config(layers):
    return DeBERTaV2Configuration(num_hidden_layers=layers) if layers == LAYERS else \
        DeBERTaV2Configuration(num_hidden_layers=layers, vocab_size=LAYER_VOCAB)


def _weights(layers):
    """Random-init weights with the checkpoint's names: linears and embeddings N(0, 0.02), gamma 1 + N(0, 0.02)."""
    g = _generator(1234)
    out = {}
    for key, shape in weight_shapes(_config(layers)).items():
        out[key] = _normal(g, shape, 0.02, 1.0 if "LayerNorm.weight" in key else 0.0)
    return out


_MODELS = {}  # a program loads its model once and serves every request with it
_KERNELS = []


def _model(layers):
    if layers not in _MODELS:
        host = {k: v.cpu().numpy() for k, v in _weights(layers).items()}
        _MODELS[layers] = GLiNERDecideClassifier(host, _config(layers))
    return _MODELS[layers]


def _kernels():
    if not _KERNELS:
        _KERNELS.append(FusedKernels())
    return _KERNELS[0]


def _classify_inputs(case, seed):
    """Token rows as the front end lays them out: [CLS], the label markers near the start, text, [SEP], padding."""
    r = np.random.default_rng([int(seed), 5])
    B, L, Hh, O = case["batch"], case["seq_len"], case["tasks"], case["labels"]
    lengths = _lengths(seed, case)
    ids = np.zeros((B, L), np.int32)
    mask = np.zeros((B, L), np.float16)
    for b in range(B):
        n = int(lengths[b])
        ids[b, :n] = r.integers(1000, 128000, size=n)
        ids[b, 0] = 1
        ids[b, 1:1 + Hh * O] = 128002
        ids[b, n - 1] = 2
        mask[b, :n] = 1
    markers = np.tile(np.arange(1, 1 + Hh * O, dtype=np.int32).reshape(1, Hh, O), (B, 1, 1))
    return ids, mask, markers, np.ones((B, Hh, O), np.float32), int(lengths.sum())


def _bucket_index(n):
    """The relative index of every distance q - k, [n, n]: linear up to 128, logarithmic to 511, clipped to 512 rows."""
    r = torch.arange(n)[:, None] - torch.arange(n)[None, :]
    a = r.abs().to(torch.float64)
    log = torch.ceil(torch.log(a.clamp(min=1) / 128) / math.log(511 / 128) * 127 - 1e-6) + 128
    bucket = torch.where(a <= 128, a, log) * torch.sign(r)
    return (bucket.to(torch.int64) + 256).clamp(0, 511)


def _attention_inputs(case, seed, values):
    g = _generator(seed)
    B, L = case["batch"], case["seq_len"]
    q = _normal(g, (B, HEADS, L, HEAD_DIM))
    k = _normal(g, (B, HEADS, L, HEAD_DIM))
    v = _normal(g, (B, HEADS, L, HEAD_DIM)) if values else None
    pk = _normal(g, (HEADS, POSITIONS, HEAD_DIM))
    pq = _normal(g, (HEADS, POSITIONS, HEAD_DIM))
    lengths = torch.from_numpy(_lengths(seed, case)).cuda()
    valid = torch.arange(L, device="cuda")[None, :] < lengths[:, None]
    return q, k, v, pk, pq, valid


def prepare(case, seed):
    kind = case["kind"]
    if kind == "classify":
        ids, mask, markers, marker_mask, total = _classify_inputs(case, seed)
        model = _model(LAYERS)
        inp = DecisionInput(ids, mask, markers, marker_mask)
        if case["host"]:
            return {"kind": "classify_host", "model": model, "input": inp}
        return {"kind": kind, "model": model, "args": inp.to_device(), "total": total}
    if kind == "layer":
        g = _generator(seed)
        B, L = case["batch"], case["seq_len"]
        mask = np.arange(L)[None, :] < _lengths(seed, case)[:, None]
        return {"kind": kind, "model": _model(1), "hidden": _normal(g, (B, L, HIDDEN)),
                "mask": torch.from_numpy(mask).cuda().to(torch.float16)}
    if kind == "linear":
        g = _generator(seed)
        rows = case["gather_from"] or case["m"]
        s = {"kind": kind, "fk": _kernels(), "x": _normal(g, (rows, case["k"])),
             "w": _normal(g, (case["n"], case["k"]), 0.02), "b": _normal(g, (case["n"],), 0.02), "rows": None,
             "epilogue": case["epilogue"]}
        if case["gather_from"]:
            s["rows"] = torch.randperm(rows, generator=g, device="cuda")[:case["m"]].sort().values.to(torch.int32)
        return s
    if kind == "ln":
        g = _generator(seed)
        return {"kind": kind, "fk": _kernels(), "x": _normal(g, (case["rows"], HIDDEN)),
                "res": _normal(g, (case["rows"], HIDDEN)), "g": _normal(g, (HIDDEN,), 0.1, 1.0),
                "b": _normal(g, (HIDDEN,), 0.1), "round_sum": case["round_sum"]}
    if kind == "attention":
        q, k, v, pk, pq, valid = _attention_inputs(case, seed, True)
        return {"kind": kind, "fk": _kernels(), "q": q, "k": k, "v": v, "pk": pk, "pq": pq,
                "mask": valid.to(torch.float16), "output": case["output"], "score": case["score"]}
    # index tensors: the model's relative positions, one table for every head, as the classifier's cache holds them
    q, k, v, pk, pq, valid = _attention_inputs(case, seed, kind == "fused")
    c2p = _bucket_index(case["seq_len"]).to(torch.int32).cuda()
    p2c = c2p.t().contiguous()  # p2c[k, q] = idx(q - k)
    key_mask = torch.where(valid, 0.0, -65504.0).to(torch.float16)
    H = HEADS
    return {"kind": kind, "fk": _kernels(), "q": q, "k": k, "v": v, "pk": pk, "pq": pq, "mask": key_mask,
            "c2p": c2p.expand(H, -1, -1).contiguous(), "p2c": p2c.expand(H, -1, -1).contiguous(),
            "scale": 1.0 / math.sqrt(3 * HEAD_DIM), "shape": (case["batch"], H, case["seq_len"])}


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind == "classify_host":
        return state["model"].classify(state["input"]).logits
    if kind == "classify":
        return state["model"].classify_device(*state["args"], total_tokens=state["total"])
    if kind == "layer":
        return state["model"].layer_forward(0, state["hidden"], state["mask"])
    fk = state["fk"]
    if kind == "linear":
        return fk.linear(state["x"], state["w"], state["b"], state["epilogue"], rows=state["rows"])
    if kind == "ln":
        return fk.residual_layer_norm(state["x"], state["res"], state["g"], state["b"], EPS,
                                      round_sum_f16=state["round_sum"])
    if kind == "attention":
        return fk.deberta_attention(state["q"], state["k"], state["v"], state["pk"], state["pq"], state["mask"],
                                    output=state["output"], score=state["score"])
    B, H, L = state["shape"]
    if kind == "bias":
        return fk.relative_bias(state["q"], state["k"], state["pk"], state["pq"], state["c2p"], state["p2c"],
                                state["mask"], state["scale"], B, H, L, HEAD_DIM, POSITIONS)
    return fk.fused_attention(state["q"], state["k"], state["v"], state["pk"], state["pq"], state["c2p"],
                              state["p2c"], state["mask"], state["scale"], B, H, L, HEAD_DIM, POSITIONS)


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _mean_length(case):
    return 0.5 * (case["min_len"] + case["seq_len"])


def _layer_work(tokens, queries, keys):
    """One layer on `tokens` rows, each of `queries` positions attending `keys` of them on average."""
    weights = 4 * HIDDEN * HIDDEN + 2 * HIDDEN * FFN
    pairs = tokens * keys * HIDDEN
    return 2.0 * tokens * weights + 2.0 * 2 * pairs, 2.0 * weights + 2.0 * 2 * POSITIONS * HIDDEN


def work(case):
    kind = case["kind"]
    C = HIDDEN
    if kind == "classify":
        n = _mean_length(case)
        tokens = case["batch"] * n
        flops, weights = _layer_work(tokens, n, n)
        markers = case["batch"] * case["tasks"] * case["labels"]
        return {"flops": LAYERS * flops + 2.0 * markers * C * CLS_HIDDEN,
                "bytes": LAYERS * weights + 2.0 * tokens * C + 2.0 * C * CLS_HIDDEN}
    if kind == "layer":
        tokens = case["batch"] * case["seq_len"]
        flops, weights = _layer_work(tokens, case["seq_len"], _mean_length(case))
        return {"flops": flops, "bytes": weights + 2.0 * 2 * tokens * C}
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"flops": 2.0 * m * n * k, "bytes": 2.0 * (m * k + n * k + m * n + n)}
    if kind == "ln":
        return {"flops": 8.0 * case["rows"] * C, "bytes": 2.0 * 3 * case["rows"] * C + 4.0 * C}
    B, L = case["batch"], case["seq_len"]
    n = _mean_length(case) if case["kind"] != "bias" else L
    rows, tables = B * HEADS * L * HEAD_DIM, 2 * HEADS * POSITIONS * HEAD_DIM
    pairs = B * HEADS * L
    if kind == "attention":
        dots = 2 if case["output"] == "context" else 1  # q.k, and P.V
        out = rows if case["output"] == "context" else pairs * L
        return {"flops": 2.0 * dots * pairs * n * HEAD_DIM,
                "bytes": 2.0 * ((1 + dots * n / L) * rows + tables + out + B * L)}
    index = 2 * HEADS * L * L
    if kind == "bias":
        return {"flops": 2.0 * 2 * pairs * L * HEAD_DIM,
                "bytes": 2.0 * (2 * rows + tables + pairs * L + B * L) + 4.0 * index}
    return {"flops": 2.0 * 4 * pairs * n * HEAD_DIM,
            "bytes": 2.0 * ((2 + 2 * n / L) * rows + tables + B * L) + 4.0 * index}


def tolerance(case):
    # Measured against `exact` over the listed cases and 30 drawn ones, times about four.
    kind = case["kind"]
    if kind == "classify":  # 24 layers of fp16 roundings
        return {"rel": 1e-2, "max": 4e-2}
    if kind == "layer":  # fp16 at every operation's output, two LayerNorms
        return {"rel": 2e-3, "max": 1.2e-2}
    if kind == "linear":  # one fp16 rounding (two with an activation) of an fp32 sum
        return {"rel": 1.3e-3, "max": 4e-3}
    if kind == "ln":
        return {"rel": 1.3e-3, "max": 4.5e-3}
    if kind == "attention":  # the bias chain rounds to fp16 four times
        return {"rel": 2.5e-3, "max": 2e-2}
    return {"rel": 8e-4, "max": 2e-3}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _f64(x):
    return x.to(torch.float64)


def _ln64(x, g, b):
    mean = x.mean(-1, keepdim=True)
    var = ((x - mean) ** 2).mean(-1, keepdim=True)
    return (x - mean) / torch.sqrt(var + EPS) * g + b


def _scores64(q, k, pk, pq, c2p, p2c, content):
    """((q.k if content) + q.pk[c2p[q, k]] + k.pq[p2c[k, q]]) / sqrt(3 D) of one row, [H, L, L]; c2p, p2c [L, L]."""
    H, L, _ = q.shape
    out = torch.gather(q @ pk.transpose(1, 2), 2, c2p.expand(H, L, L))
    out += torch.gather(k @ pq.transpose(1, 2), 2, p2c.expand(H, L, L)).transpose(1, 2)
    if content:
        out += q @ k.transpose(1, 2)
    return out / math.sqrt(3 * HEAD_DIM)


def _softmax64(scores, valid):
    return torch.softmax(scores.masked_fill(~valid[None, None, :], -math.inf), -1)


def _layer64(x, w, prefix, rel, valid):
    """One encoder layer on x [B, L, C] in 64 bits; w gives a weight by its name, rel the normed relative table."""
    B, L, C = x.shape
    att = prefix + ".attention.self."

    def heads(t):
        return t.reshape(-1, HEADS, HEAD_DIM).transpose(0, 1)

    def linear(t, name):
        return t @ w(name + ".weight").t() + w(name + ".bias")

    idx = _bucket_index(L).cuda()
    pk, pq = heads(linear(rel, att + "key_proj")), heads(linear(rel, att + "query_proj"))
    ctx = torch.empty_like(x)
    for b in range(B):
        q, k, v = (heads(linear(x[b], att + n + "_proj")) for n in ("query", "key", "value"))
        p = _softmax64(_scores64(q, k, pk, pq, idx, idx.t(), True), valid[b])
        ctx[b] = (p @ v).transpose(0, 1).reshape(L, C)
    out = prefix + ".attention.output."
    x = _ln64(linear(ctx, out + "dense") + x, w(out + "LayerNorm.weight"), w(out + "LayerNorm.bias"))
    y = torch.nn.functional.gelu(linear(x, prefix + ".intermediate.dense"))
    out = prefix + ".output."
    return _ln64(linear(y, out + "dense") + x, w(out + "LayerNorm.weight"), w(out + "LayerNorm.bias"))


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        s = prepare(case, seed)
        x = s["x"] if s["rows"] is None else s["x"][s["rows"].long()]
        y = _f64(x) @ _f64(s["w"]).t() + _f64(s["b"])
        return torch.nn.functional.gelu(y) if case["epilogue"] == "gelu" else \
            torch.relu(y) if case["epilogue"] == "relu" else y
    if kind == "ln":
        s = prepare(case, seed)
        return _ln64(_f64(s["x"]) + _f64(s["res"]), _f64(s["g"]), _f64(s["b"]))
    if kind in ("attention", "bias", "fused"):
        s = prepare(case, seed)
        B, L = case["batch"], case["seq_len"]
        idx = _bucket_index(L).cuda()
        pk, pq = _f64(s["pk"]), _f64(s["pq"])
        out = []
        for b in range(B):
            valid = s["mask"][b] > (0 if kind == "attention" else -60000)
            t = _scores64(_f64(s["q"][b]), _f64(s["k"][b]), pk, pq, idx, idx.t(), kind != "bias")
            if kind == "bias":
                out.append(t.masked_fill(~valid[None, None, :], -65504.0))
                continue
            p = _softmax64(t, valid)
            if kind == "attention" and case["output"] == "probs":
                out.append(p)
                continue
            o = (p @ _f64(s["v"][b])).transpose(0, 1)
            out.append(o.reshape(L, HIDDEN) if kind == "attention" else o)
        return torch.stack(out)

    layers = LAYERS if kind == "classify" else 1
    weights = _weights(layers)

    def w(name):
        return _f64(weights[name])

    enc = "encoder.encoder."
    rel = _ln64(w(enc + "rel_embeddings.weight"), w(enc + "LayerNorm.weight"), w(enc + "LayerNorm.bias"))
    if kind == "layer":
        s = prepare(case, seed)
        return _layer64(_f64(s["hidden"]), w, enc + "layer.0", rel, s["mask"] > 0)
    ids, mask, markers, _, _ = _classify_inputs(case, seed)
    valid = torch.from_numpy(mask).cuda() > 0
    emb = "encoder.embeddings."
    x = _f64(weights[emb + "word_embeddings.weight"][torch.from_numpy(ids).cuda().long()])
    x = _ln64(x, w(emb + "LayerNorm.weight"), w(emb + "LayerNorm.bias")) * valid[..., None]
    for i in range(layers):
        x = _layer64(x, w, enc + "layer.%d" % i, rel, valid)
    B = case["batch"]
    rows = x[torch.arange(B, device="cuda")[:, None], torch.from_numpy(markers.reshape(B, -1)).cuda().long()]
    inner = torch.relu(rows @ w("classifier.0.weight").t() + w("classifier.0.bias"))
    logits = inner @ w("classifier.2.weight").t() + w("classifier.2.bias")
    return logits.reshape(B, case["tasks"], case["labels"])
