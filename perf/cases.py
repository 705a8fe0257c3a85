"""The workloads this framework is measured on.

Five ways a program uses it, all through the public entry points:

  step        one batch of the op-level forward: `build_tree` fills the node rows of K / V, then
              `hierarchical_attention` runs on them (inference; no autograd)
  attn_train  `hierarchical_attention` forward and backward on given K / V rows
  module      one `HierarchicalAttention` module in training: span-node update, attention over the
              updated nodes, backward into activations and weights, under autocast with fp32 weights
  lm          forward of the decoder language model (`TransformerLM`), evaluation mode
  lm_train    forward, cross-entropy and backward of the same model

The ranges: sequence lengths 64 .. 65536 (powers of two: the tree is complete), batches 1 .. 16, heads
1 .. 16, 32 .. 128 channels per head, window radii 1 .. 32, causal or not, bf16 / fp16 / fp32.
"""
import math

import torch
import torch.nn.functional as F

import sparseattention_amd as sa

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}


def listed():
    op = dict(kind="step", causal=True)
    lm = dict(kind="lm", dtype="bf16", vocab=50257, dim=512, heads=8, ff=2048, layers=6, window=16)
    return [
        # the smallest op call: a few thousand head-queries in fp32, all launches and host time
        dict(op, name="step_small_fp32", dtype="fp32", batch=2, heads=4, leaves=256, head_dim=32, window=8),
        # short sequences in a batch (bench.py's B16 H8 N512 configuration)
        dict(op, name="step_short_bf16", dtype="bf16", batch=16, heads=8, leaves=512, head_dim=64, window=8),
        # the headline configuration of bench.py
        dict(op, name="step_headline_bf16", dtype="bf16", batch=8, heads=8, leaves=2048, head_dim=64, window=16),
        # an encoder's pass: no causal mask, odd batch, 12 heads, a window radius that is no power of two
        dict(op, name="step_encoder_fp16", dtype="fp16", batch=5, heads=12, leaves=1024, head_dim=64, window=13,
             causal=False),
        # a model width of 768 over 8 heads: 96 channels per head
        dict(op, name="step_head96_bf16", dtype="bf16", batch=3, heads=8, leaves=2048, head_dim=96, window=16),
        # the long-sequence configuration of bench.py (one document of 65536 tokens): the largest
        dict(op, name="step_long_bf16", dtype="bf16", batch=1, heads=16, leaves=65536, head_dim=128, window=32),
        # the op in a training step at the headline shape
        dict(kind="attn_train", name="attn_train_bf16", dtype="bf16", batch=8, heads=8, leaves=2048, head_dim=64,
             window=16, causal=True),
        # the same in full precision, a small odd batch
        dict(kind="attn_train", name="attn_train_fp32", dtype="fp32", batch=3, heads=8, leaves=1024, head_dim=64,
             window=16, causal=True),
        # one module of the pre-training configuration (width 768, 12 heads, 8 x 2048 tokens, fp16 autocast)
        dict(kind="module", name="module_train_amp", dtype="fp16", batch=8, leaves=2048, dim=768, heads=12, window=16),
        # scoring one short prompt: the latency of a single sequence through six layers
        dict(lm, name="lm_prompt", batch=1, leaves=256),
        # the language-model configuration of bench.py
        dict(lm, name="lm_forward", batch=8, leaves=4096),
        # a training step of a small model of the same width
        dict(lm, name="lm_train", kind="lm_train", layers=2, batch=4, leaves=1024),
    ]


# ---------------------------------------------------------------------------------------- draws
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["attn_train"] * 4 + ["module"] * 2 + ["lm"] * 2 + ["lm_train"])
    while True:
        causal = rng.random() < 0.75
        if kind in ("step", "attn_train"):
            c = dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"]), causal=causal,
                     batch=_log_int(rng, 1, 16), heads=rng.randint(1, 16), leaves=2 ** rng.randint(6, 16),
                     head_dim=rng.choice([32, 48, 64, 64, 64, 80, 96, 128, 128]), window=rng.randint(1, 32))
            size = c["batch"] * c["heads"] * c["leaves"] * c["head_dim"] * BYTES[c["dtype"]]
            # at least the smallest listed step, at most the long-sequence one (a third of it in
            # training; head sizes between the powers of two are drawn smaller)
            most = 2 ** 28 if kind == "step" else 2 ** 28 // 3
            if 2 ** 18 <= size <= (most if c["head_dim"] in (32, 64, 128) else most // 12):
                return c
        elif kind == "module":
            hd = rng.choice([32, 64, 64, 96, 128])
            c = dict(kind=kind, dtype=rng.choice(["bf16", "fp16"]), batch=rng.randint(1, 8), heads=rng.randint(2, 16),
                     leaves=2 ** rng.randint(6, 12), window=rng.randint(4, 32))
            c["dim"] = c["heads"] * hd
            if 256 <= c["dim"] <= 1024 and c["batch"] * c["leaves"] <= 2 ** 14:
                return c
        else:
            hd = rng.choice([32, 64, 64, 128])
            # (training in plain fp16, without an optimizer's loss scaling, is nobody's use: bf16 there)
            c = dict(kind=kind, dtype=rng.choice(["bf16", "fp16"] if kind == "lm" else ["bf16"]), vocab=_log_int(rng, 1000, 50257),
                     heads=rng.randint(2, 12), layers=rng.randint(2, 6) if kind == "lm" else rng.randint(1, 3),
                     batch=rng.randint(1, 8), leaves=2 ** rng.randint(6, 12), window=rng.randint(4, 32))
            c["dim"] = c["heads"] * hd
            c["ff"] = 4 * c["dim"]
            tokens = c["batch"] * c["leaves"]
            if 256 <= c["dim"] <= 768 and tokens * c["layers"] <= (2 ** 17 if kind == "lm" else 2 ** 13):
                return c


# ---------------------------------------------------------------------------------------- inputs
def prepare(case, seed):
    g = torch.Generator(DEV).manual_seed(seed)
    dt, kind = DTYPES[case["dtype"]], case["kind"]
    B, N = case["batch"], case["leaves"]

    def normal(*shape, dtype=dt, scale=1.0):
        return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).mul_(scale).to(dtype)

    s = {"kind": kind, "window": case["window"]}
    if kind in ("step", "attn_train"):
        H, D = case["heads"], case["head_dim"]
        s["tables"] = sa.build_tree_topology(N, case["causal"], device=DEV)
        s["mask"] = s["tables"]["forward_mask"] if case["causal"] else None
        s["q"] = normal(B, N, H, D)
        # leaf rows first, then the node rows level by level
        s["k"], s["v"] = normal(B, 2 * N - 1, H, D), normal(B, 2 * N - 1, H, D)
        if kind == "step":
            s["qp"], s["kp"], s["vp"] = (normal(B, N - 1, H, D) for _ in range(3))
        else:
            s["dout"] = normal(B, N, H, D)
            for n in ("q", "k", "v"):
                s[n].requires_grad_(True)
        return s
    torch.manual_seed(seed)
    if kind == "module":
        dim = case["dim"]
        with torch.device(DEV):
            s["net"] = sa.HierarchicalAttention(dim, case["heads"], dropout=0.0, window_size=case["window"]).train()
        s["amp"] = dt
        s["x"] = normal(B, N, dim, dtype=torch.float32).requires_grad_(True)
        s["y"] = normal(B, N - 1, dim, dtype=torch.float32).requires_grad_(True)
        s["dx"], s["dy"] = normal(B, N, dim, dtype=torch.float32), normal(B, N - 1, dim, dtype=torch.float32)
        s["mask"] = torch.ones(1, 1, 1, 1, dtype=torch.bool, device=DEV)
        return s
    with torch.device(DEV):
        net = sa.TransformerLM(case["vocab"], case["dim"], case["heads"], case["ff"], case["layers"], dropout=0.0,
                               window_size=case["window"], activation="gelu", max_len=N)
    s["net"] = net.to(dt).train(kind == "lm_train")
    s["tokens"] = torch.randint(0, case["vocab"], (B, N), generator=g, device=DEV)
    if kind == "lm_train":
        s["targets"] = torch.randint(0, case["vocab"], (B * N,), generator=g, device=DEV)
    return s


# ---------------------------------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "step":
        t, N = s["tables"], s["q"].shape[1]
        with torch.no_grad():
            k, v = s["k"], s["v"]
            sa.build_tree(s["qp"], s["kp"], s["vp"], k[:, :N], v[:, :N], out=k[:, N:], out2=v[:, N:])
            out = sa.hierarchical_attention(s["q"], k, v, t["forward_idx"], t["backward_gather"], s["mask"], s["window"])
        return out, k[:, N:], v[:, N:]
    if kind == "attn_train":
        t, q, k, v = s["tables"], s["q"], s["k"], s["v"]
        q.grad = k.grad = v.grad = None
        out = sa.hierarchical_attention(q, k, v, t["forward_idx"], t["backward_gather"], s["mask"], s["window"])
        out.backward(s["dout"])
        return out.detach(), q.grad, k.grad, v.grad
    net = s["net"]
    if kind == "module":
        net.zero_grad(set_to_none=True)
        x, y = s["x"], s["y"]
        x.grad = y.grad = None
        with torch.autocast("cuda", dtype=s["amp"]):
            nodes = net.cross_update_Y(x, y)
            out = net(x, x, x, y=nodes, mask=s["mask"])
        torch.autograd.backward([out, nodes], [s["dx"].to(out.dtype), s["dy"].to(nodes.dtype)])
        return out.detach(), nodes.detach(), x.grad, y.grad, [p.grad for p in net.parameters()]
    if kind == "lm":
        with torch.no_grad():
            return net(s["tokens"])
    net.zero_grad(set_to_none=True)
    logits = net(s["tokens"])
    loss = F.cross_entropy(logits.float().view(-1, logits.shape[-1]), s["targets"])
    loss.backward()
    return logits.detach(), [p.grad for p in net.parameters() if p.grad is not None]


# ---------------------------------------------------------------------------------------- floors
def work(case):
    """Bytes that have to move (each input read once, each output written once) and operations of one
    pass.  A query attends to its window and to one node per level; half of the node slots are dead
    under the causal mask, and so is the right half of the window."""
    kind, B, N, H = case["kind"], case["batch"], case["leaves"], case["heads"]
    D = case["head_dim"] if "head_dim" in case else case["dim"] // H
    e, L, R = BYTES[case["dtype"]], N.bit_length() - 1, case["window"]
    M = 2 * N - 1
    row = B * H * D
    keys = (R + 1 + L / 2) if case.get("causal", True) else (2 * R + 1 + L)
    attn = 4.0 * row * N * keys          # q.k and p.v of every attended key
    tree = 12.0 * row * (N - 1)          # three keys per node, both products
    if kind == "step":
        # queries, leaves, the nodes' own q / k / v in; output rows and both copies of the nodes out
        return {"bytes": float(e * row * (N + 2 * N + 3 * (N - 1) + N + 2 * (N - 1))), "flops": attn + tree}
    if kind == "attn_train":
        # q, k, v, dout in; out, dq, dk, dv out
        return {"bytes": float(e * row * (4 * N + 4 * M)), "flops": 3.5 * attn}
    T, d = B * N, case["dim"]
    nodes = B * (N - 1)
    # projections of one layer's attention: q, k, v of the nodes, k, v of every level's children,
    # out_proj_y; q, k, v of the leaves, k, v of the nodes, out_proj_x
    proj = 2.0 * d * d * (3 * nodes + 2 * (T + nodes) + nodes + 3 * T + 2 * nodes + T)
    if kind == "module":
        # activations and their gradients in fp32, weights and their gradients in fp32
        acts = 4.0 * (T + nodes) * d
        weights = 4.0 * (8 * d * d + 2 * d)
        return {"bytes": 4 * acts + 2 * weights, "flops": 3 * (proj + tree) + 3.5 * attn}
    V, ff, layers = case["vocab"], case["ff"], case["layers"]
    weights = e * (V * d + layers * (8 * d * d + 2 * d * ff))
    logits = e * T * V
    flops = layers * (proj + tree + attn + 4.0 * T * d * ff) + 2.0 * T * d * V
    if kind == "lm":
        return {"bytes": float(weights + logits), "flops": flops}
    return {"bytes": float(2 * weights + 3 * logits), "flops": 3 * flops}


def tolerance(case):
    """About four times what the path differs from the same computation at a higher precision on the
    same inputs: the 16-bit paths from this package's fp32 one (bf16: ops 2.4e-3, module 6.2e-3, model
    9e-3; fp16: ops 3e-4, module 8e-4, model 8e-4), the fp32 ops from fp64 (3e-7)."""
    op = case["kind"] in ("step", "attn_train")
    if case["dtype"] == "fp32":
        return {"rel": 1.2e-6, "max": 4e-5}
    if case["dtype"] == "fp16":
        return {"rel": 1.2e-3, "max": 0.05} if op else {"rel": 3.2e-3, "max": 0.05}
    return {"rel": 1e-2, "max": 0.25} if op else {"rel": 0.025, "max": 0.4}
