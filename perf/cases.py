"""The work that a user of the quantised Dense path has it do, as cases to be timed.

Every case goes through the public entry points of gomlx_amd.nn on GPU tensors.  Kinds:

* dense      one projection, ``quantized_dense`` (optionally with bias and activation, or behind an RMS norm);
* layer      the seven projections of one decoder layer as a model calls them: q / k / v behind the input norm
             in one submission, the output projection with its residual, the gated feed-forward front behind
             the second norm, the down projection with its residual.  Attention is outside this path: the
             query projection stands in for its result, so that the four calls depend on each other;
* gated      the gated feed-forward front alone;
* dequantize the exact dequantisation of a whole matrix;
* gather     rows of a quantised embedding table.

A state holds the weights of its matrices as a program holds a loaded model; activations come from the seed.
"""
from __future__ import annotations

import math

import torch

from gomlx_amd import ggml, nn

TYPES = {"Q8_0": ggml.Q8_0, "Q4_0": ggml.Q4_0, "Q4_K": ggml.Q4_K, "Q6_K": ggml.Q6_K, "IQ4_NL": ggml.IQ4_NL}
ACTS = {"none": nn.Activation.NONE, "gelu": nn.Activation.GELU, "silu": nn.Activation.SILU, "relu": nn.Activation.RELU}
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}

# Standard deviation of a weight per unit of the block scale d, for codes that are uniform over their range (IQ4_NL: over
# its code book; Q4_K: centred code times a 6-bit sub-block scale; Q6_K: code times an int8 scale).
_SPREAD = {"Q8_0": 73.6, "Q4_0": 4.61, "Q4_K": 170.0, "Q6_K": 1370.0, "IQ4_NL": 70.0}


def listed():
    return [
        # One token through one projection: the smallest call, where latency and launches count.
        dict(name="dense_q8_0_rows1", kind="dense", type="Q8_0", dtype="f32", rows=1, k=4096, n=4096, act="none", bias=False, norm=False),
        # One token through a wide projection (the up projection of a feed-forward block).
        dict(name="dense_q4_0_rows1", kind="dense", type="Q4_0", dtype="f32", rows=1, k=4096, n=14336, act="none", bias=False, norm=False),
        # A decode batch through a long contraction (the down projection).
        dict(name="dense_q4_k_rows32", kind="dense", type="Q4_K", dtype="f32", rows=32, k=14336, n=4096, act="none", bias=False, norm=False),
        # A prompt through one projection in bfloat16.
        dict(name="dense_q8_0_bf16_rows2048", kind="dense", type="Q8_0", dtype="bf16", rows=2048, k=4096, n=4096, act="none", bias=False, norm=False),
        # A ragged call: K not a multiple of 256, odd row count, N off every tile, with bias and activation.
        dict(name="dense_iq4_nl_ragged", kind="dense", type="IQ4_NL", dtype="f32", rows=77, k=2080, n=1500, act="gelu", bias=True, norm=False),
        # Logits of a few sequences: final norm and output head over a large vocabulary, bfloat16 activations.
        dict(name="head_q6_k_bf16_rows4", kind="dense", type="Q6_K", dtype="bf16", rows=4, k=4096, n=128256, act="none", bias=False, norm=True),
        # A decoder layer: one sequence; a decode batch of eight; a large decode batch or a short prompt; a prompt.
        dict(name="layer_q4_k_rows1", kind="layer", type="Q4_K", dtype="f32", rows=1, k=4096, kv=1024, n=14336),
        dict(name="layer_q4_k_rows8", kind="layer", type="Q4_K", dtype="f32", rows=8, k=4096, kv=1024, n=14336),
        dict(name="layer_q4_k_rows128", kind="layer", type="Q4_K", dtype="f32", rows=128, k=4096, kv=1024, n=14336),
        dict(name="layer_q4_k_rows512", kind="layer", type="Q4_K", dtype="f32", rows=512, k=4096, kv=1024, n=14336),
        # Weights back to float32, as a tool or a fallback path asks for them.
        dict(name="dequantize_q4_k", kind="dequantize", type="Q4_K", dtype="f32", rows=0, k=4096, n=14336),
        # The embedding of a prompt.
        dict(name="gather_q8_0_rows512", kind="gather", type="Q8_0", dtype="f32", rows=512, k=4096, n=128256),
    ]


_MAX_FLOPS = 2.2e11        # of the largest listed case (the layer at 512 rows)
_MAX_WEIGHTS = 1.1e9       # values in the matrices of a case


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    while True:
        kind = rng.choice(("dense", "dense", "dense", "layer", "layer", "layer", "gated", "gated", "dequantize", "gather"))
        t = rng.choice(("Q4_K", "Q4_K", "Q8_0", "Q4_0", "Q6_K", "IQ4_NL"))
        super_block = t in ("Q4_K", "Q6_K")
        dtype = rng.choice(("f32", "f32", "bf16"))
        rows = _log(rng, 1, 2048)
        if kind == "layer":  # hidden sizes in whole heads of 128
            k = 256 * _log(rng, 4, 20)
            c = dict(kind=kind, type=t, dtype="f32", rows=rows, k=k, kv=128 * max(1, k // 512), n=256 * _log(rng, 8, 60))
        elif kind == "gated":
            c = dict(kind=kind, type=t, dtype=dtype, rows=rows, k=256 * _log(rng, 4, 32), n=_log(rng, 1024, 16384), act=rng.choice(("silu", "silu", "gelu")), norm=rng.random() < 0.7)
        elif kind == "dense":
            k = 256 * _log(rng, 4, 60) if super_block or rng.random() < 0.7 else 32 * _log(rng, 32, 480)
            c = dict(kind=kind, type=t, dtype=dtype, rows=rows, k=k, n=_log(rng, 512, 32768), act=rng.choice(("none", "none", "gelu", "silu", "relu")),
                     bias=rng.random() < 0.3, norm=rng.random() < 0.3)
        else:
            c = dict(kind=kind, type=t, dtype="f32", rows=0 if kind == "dequantize" else _log(rng, 1, 4096), k=256 * _log(rng, 4, 56),
                     n=_log(rng, 1024, 16384) if kind == "dequantize" else _log(rng, 30000, 130000))
        if work(c)["flops"] <= _MAX_FLOPS and sum(n * k for n, k in _matrices(c)) <= _MAX_WEIGHTS:
            return c


def _matrices(c):
    """(rows, columns) of every weight matrix of the case, in the order in which the state holds them."""
    k, n = c["k"], c["n"]
    if c["kind"] == "layer":
        return [(k, k), (c["kv"], k), (c["kv"], k), (k, k), (n, k), (n, k), (k, n)]
    return [(n, k), (n, k)] if c["kind"] == "gated" else [(n, k)]


def _weights(t, N, K, gen):
    """Random GGML blocks [N, bytesPerRow]: codes uniform over their range, block scales |N(0, s)| with s such that the
    weights have a standard deviation of about 1 / sqrt(K).  The minima of Q4_K centre the codes of their sub-blocks, as a
    quantiser of weights around zero leaves them."""
    bpb, vpb = ggml.bytes_per_block(TYPES[t]), ggml.values_per_block(TYPES[t])
    nb = N * (K // vpb)
    dev = gen.device
    out = torch.randint(0, 256, (nb, bpb), dtype=torch.uint8, device=dev, generator=gen)

    def halves(v):
        return v.to(torch.float16).view(torch.uint8).view(nb, 2)

    d = torch.randn(nb, device=dev, generator=gen).abs() / (math.sqrt(K) * _SPREAD[t])
    if t == "Q6_K":
        out[:, 208:210] = halves(d)
    else:
        out[:, 0:2] = halves(d)
        if t == "Q4_K":  # minimum = scale code of its sub-block, dmin = mean code * d
            out[:, 2:4] = halves(7.5 * d)
            out[:, 8:12] = out[:, 4:8]
            out[:, 12:16] = (out[:, 12:16] & 15) * 17
        elif t == "Q8_0":  # codes in [-127, 127]
            q = out[:, 2:]
            q[q == 0x80] = 0x81
    return out.view(N, K // vpb * bpb)


def prepare(case, seed):
    c = dict(case)
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    st = dict(case=c, quant=nn.Quantization(ggml_type=TYPES[c["type"]]), w=[_weights(c["type"], n, k, gen) for n, k in _matrices(c)])
    if c["kind"] == "gather":
        st["idx"] = torch.randint(0, c["n"], (c["rows"], 1), dtype=torch.int32, device=dev, generator=gen)
    elif c["kind"] != "dequantize":
        st["x"] = torch.randn(c["rows"], c["k"], device=dev, generator=gen).to(DTYPES[c["dtype"]])
        gains = [1.0 + 0.1 * torch.randn(c["k"], device=dev, generator=gen) for _ in range(2)]
        st["norms"] = [nn.RMSNorm(gain=g, epsilon=1e-5) for g in gains]
        st["bias"] = 0.1 * torch.randn(c["n"], device=dev, generator=gen) if c.get("bias") else None
    return st


def run(st):
    c, w, q = st["case"], st["w"], st["quant"]
    kind = c["kind"]
    if kind == "dequantize":
        return nn.dequantize(w[0], q.ggml_type)
    if kind == "gather":
        return nn.quantized_gather(w[0], st["idx"], q)
    x, norms = st["x"], st["norms"]
    if kind == "dense":
        return nn.quantized_dense(x, w[0], q, st["bias"], ACTS[c["act"]], norm=norms[0] if c["norm"] else None)
    if kind == "gated":
        return nn.gated_feed_forward(x, w[0], w[1], q, ACTS[c["act"]], norm=norms[0] if c["norm"] else None)
    query, key, value = nn.quantized_dense_batch([(x, w[i], q, None, None) for i in range(3)], norm=norms[0])
    h = nn.quantized_dense(query, w[3], q, residual=x)
    f = nn.gated_feed_forward(h, w[4], w[5], q, nn.Activation.SILU, norm=norms[1])
    y = nn.quantized_dense(f, w[6], q, residual=h)
    return query, key, value, y


def work(case):
    c = case
    mats = _matrices(c)
    t = TYPES[c["type"]]
    weight_bytes = sum(n * ggml.row_bytes(t, k) for n, k in mats)
    if c["kind"] == "dequantize":
        return {"bytes": weight_bytes + 4 * c["n"] * c["k"], "flops": 2 * c["n"] * c["k"]}
    if c["kind"] == "gather":
        return {"bytes": c["rows"] * (ggml.row_bytes(t, c["k"]) + 4 * c["k"] + 4), "flops": 2 * c["rows"] * c["k"]}
    xb = 4 if c["dtype"] == "f32" else 2
    out = 2 * c["k"] + 2 * c["kv"] if c["kind"] == "layer" else c["n"]
    return {"bytes": weight_bytes + c["rows"] * (c["k"] * xb + out * 4), "flops": 2 * c["rows"] * sum(n * k for n, k in mats)}


def tolerance(case):
    c = case
    if c["kind"] in ("dequantize", "gather"):
        return "exact"
    # About four times what a contraction in 64 bits on the dequantised weights differs by (figures: relative 2-norm).
    if c["dtype"] == "bf16" and c["kind"] == "dense" and c["rows"] > 16 and not c["norm"]:
        return {"rel": 7e-3}    # 1.7e-3: weights rounded to bfloat16 operands
    if c["rows"] <= 2:
        return {"rel": 1.2e-4}  # 2.1e-5 to 3.0e-5: 16-bit fixed-point activations
    if c["type"] == "Q4_K":     # 5.2e-4 and 6.6e-4: the same, beside the larger terms that a block's minimum cancels
        return {"rel": 2.1e-3 if c["kind"] == "dense" else 2.6e-3}
    if c["kind"] == "dense":
        return {"rel": 1.2e-3}  # 2.4e-4 to 3.1e-4: float16 operands
    return {"rel": 1.7e-3}      # 4.2e-4: the same, in a product of two projections
