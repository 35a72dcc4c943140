"""The calls a program makes of this framework, one dict per case.

Every case goes through a public entry point: the norm, softmax and
cross-entropy ``kernel_fn``s, the ``torch.ops.autokernel`` ops under autograd,
``ChunkedLinearCrossEntropyLoss``, ``selective_scan_fn`` and the diagonal scan.
Inputs are made on the GPU from a seed. ``exact`` restates each path in float64
torch, without the framework.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "autokernel-halo-strix_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_SIZE = {"f32": 4, "f16": 2, "bf16": 2}


def listed():
    return [
        # one decode step of a batch of 8: the pre-attention norm, a launch and little else
        {"name": "rmsnorm_decode", "op": "rmsnorm", "dtype": "bf16", "rows": 8, "cols": 4096},
        # a block's residual add + norm over a 16k-token prefill or training batch
        {"name": "add_rmsnorm_16k", "op": "add_rmsnorm", "dtype": "bf16", "rows": 16384, "cols": 4096},
        # the same block in training, through the registered op: forward, then all gradients
        {"name": "add_rmsnorm_train", "op": "add_rmsnorm_train", "dtype": "bf16", "rows": 8192, "cols": 2048},
        # causal attention probabilities, batch 8 x 12 heads at 1024 tokens
        {"name": "softmax_causal", "op": "softmax", "dtype": "f16", "rows": 98304, "cols": 1024, "causal": True},
        # next-token probabilities over GPT-2's vocabulary, whose rows are not 16-byte aligned
        {"name": "softmax_vocab", "op": "softmax", "dtype": "f16", "rows": 4096, "cols": 50257, "causal": False},
        # training loss over materialised logits, gradient written by the forward
        {"name": "ce_fused_32k", "op": "ce", "dtype": "bf16", "rows": 4096, "vocab": 32768, "mode": "fused",
         "softcap": 0.0, "smoothing": 0.0, "z_loss": 0.0},
        # the same over GPT-2's vocabulary, gradient recomputed in the backward to save memory
        {"name": "ce_tiny_gpt2", "op": "ce", "dtype": "f16", "rows": 4096, "vocab": 50257, "mode": "tiny",
         "softcap": 0.0, "smoothing": 0.0, "z_loss": 0.0},
        # lm-head + loss of a GPT-2-sized model, a whole training step of 8 x 1024 tokens
        {"name": "lmhead_train_8k", "op": "lmhead", "dtype": "bf16", "rows": 8192, "vocab": 50304, "d": 768,
         "softcap": 0.0, "smoothing": 0.0, "train": True},
        # the small training batch of the reference's language model: 4 x 256 tokens, softcap 30
        {"name": "lmhead_train_1k", "op": "lmhead", "dtype": "bf16", "rows": 1024, "vocab": 32768, "d": 768,
         "softcap": 30.0, "smoothing": 0.0, "train": True},
        # Mamba-1 prefill of one prompt, whose length is what it is; the state goes on to decode
        {"name": "scan_prefill", "op": "scan", "dtype": "bf16", "batch": 1, "dim": 2048, "seqlen": 1777,
         "dstate": 16, "train": False},
        # Mamba-1 training step of 4 x 4096 tokens
        {"name": "scan_train", "op": "scan", "dtype": "bf16", "batch": 4, "dim": 2048, "seqlen": 4096,
         "dstate": 16, "train": True},
        # the diagonal scan of the AMADEUS block in training, through the registered op
        {"name": "diag_train", "op": "diag", "batch": 16, "seqlen": 1024, "dim": 384, "train": True},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rough(rng, n, unit):
    """n as it is one time in three, otherwise a multiple of ``unit``."""
    return n if rng.random() < 1 / 3 else max(unit, n // unit * unit)


def draw(rng):
    op = rng.choice(["rmsnorm", "add_rmsnorm", "add_rmsnorm_train", "softmax", "softmax", "ce", "ce",
                     "lmhead", "lmhead", "scan", "scan", "scan", "diag", "diag"])
    if op in ("rmsnorm", "add_rmsnorm", "add_rmsnorm_train"):
        rows = _spread(rng, 1 if op != "add_rmsnorm_train" else 64, 16384)
        cols = _rough(rng, _spread(rng, 256, 8192), 64)
        return {"op": op, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "rows": rows,
                "cols": min(cols, (1 << 26) // rows)}
    if op == "softmax":
        dtype = rng.choice(["f16", "bf16", "f32"])
        if rng.random() < 0.6:  # attention: batch x heads planes of tokens x tokens
            cols = _rough(rng, _spread(rng, 64, 4096), 64)
            planes = rng.choice([8, 12, 32, 64, 96])
            planes = max(1, min(planes, 100_000_000 // (cols * cols)))
            return {"op": op, "dtype": dtype, "rows": planes * cols, "cols": cols, "causal": True}
        cols = _rough(rng, _spread(rng, 4096, 65536), 64)
        return {"op": op, "dtype": dtype, "rows": min(_spread(rng, 8, 8192), 200_000_000 // cols),
                "cols": cols, "causal": False}
    if op == "ce":
        vocab = _rough(rng, _spread(rng, 1024, 65536), 64)
        return {"op": op, "dtype": rng.choice(["bf16", "f16", "f32"]),
                "rows": min(_spread(rng, 128, 8192), 200_000_000 // vocab), "vocab": vocab,
                "mode": rng.choice(["fused", "fused", "tiny"]), "softcap": rng.choice([0.0, 0.0, 30.0]),
                "smoothing": rng.choice([0.0, 0.0, 0.1]), "z_loss": rng.choice([0.0, 0.0, 1e-4])}
    if op == "lmhead":
        return {"op": op, "dtype": rng.choice(["bf16", "bf16", "f16"]), "rows": _spread(rng, 128, 8192),
                "vocab": _rough(rng, _spread(rng, 4096, 50304), 64), "d": rng.choice([256, 512, 640, 768]),
                "softcap": rng.choice([0.0, 30.0]), "smoothing": rng.choice([0.0, 0.0, 0.1]),
                "train": rng.random() < 0.7}
    if op == "scan":
        train = rng.random() < 0.5
        seqlen = _spread(rng, 64, 4096)
        if train:  # training batches are mostly packed to whole lengths, prompts are not
            seqlen = _rough(rng, seqlen, 64)
        return {"op": op, "dtype": rng.choice(["bf16", "bf16", "f16"]), "batch": rng.choice([1, 2, 4]),
                "dim": rng.choice([384, 768, 1536, 2048]), "seqlen": seqlen,
                "dstate": rng.choice([16, 16, 16, 64]) if not train else 16, "train": train}
    return {"op": op, "batch": rng.choice([1, 4, 8, 16]), "seqlen": _rough(rng, _spread(rng, 128, 4096), 64),
            "dim": rng.choice([128, 384, 512]), "train": rng.random() < 0.7}


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(dtype)


def _targets(g, rows, vocab):
    """Token ids, 5% of them masked with the default ignore_index."""
    t = torch.randint(0, vocab, (rows,), generator=g, device="cuda")
    return t.masked_fill(torch.rand(rows, generator=g, device="cuda") < 0.05, -100)


def _inputs(c, seed):
    g = _gen(seed)
    op = c["op"]
    dt = _DT.get(c.get("dtype"), torch.float32)
    if op in ("rmsnorm", "add_rmsnorm", "add_rmsnorm_train"):
        r, n = c["rows"], c["cols"]
        s = {"x": _randn(g, r, n, dtype=dt), "w": (1 + _randn(g, n, scale=0.02)).to(dt)}
        if op != "rmsnorm":
            s["r"] = _randn(g, r, n, dtype=dt)
        if op == "add_rmsnorm_train":
            s["gh"], s["gy"] = _randn(g, r, n, dtype=dt), _randn(g, r, n, dtype=dt)
        return s
    if op == "softmax":
        x = _randn(g, c["rows"], c["cols"], dtype=dt, scale=3.0)
        if c["causal"]:
            n = c["cols"]
            mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
            x = x.view(-1, n, n).masked_fill_(mask, float("-inf"))
        return {"x": x}
    if op == "ce":
        return {"x": _randn(g, c["rows"], c["vocab"], dtype=dt, scale=2.0), "t": _targets(g, c["rows"], c["vocab"])}
    if op == "lmhead":
        return {"h": _randn(g, c["rows"], c["d"], dtype=dt),
                "w": _randn(g, c["vocab"], c["d"], dtype=dt, scale=0.02), "t": _targets(g, c["rows"], c["vocab"])}
    if op == "scan":
        b, d, l, n = c["batch"], c["dim"], c["seqlen"], c["dstate"]
        # as the Mamba-1 block forms them: the gate is half of the input
        # projection, dt a small projection plus the softplus inverse of a step
        # size in [1e-3, 1e-1], A = -(1..N)
        xz = _randn(g, b, 2 * d, l, dtype=dt)
        step = torch.exp(torch.rand(d, generator=g, device="cuda") * math.log(100.0) + math.log(1e-3))
        s = {"u": _randn(g, b, d, l, dtype=dt), "z": xz[:, d:], "delta": _randn(g, b, d, l, dtype=dt, scale=0.5),
             "A": -torch.arange(1, n + 1, dtype=torch.float32, device="cuda").repeat(d, 1),
             "B": _randn(g, b, n, l, dtype=dt), "C": _randn(g, b, n, l, dtype=dt),
             "D": torch.ones(d, device="cuda"), "bias": step + torch.log(-torch.expm1(-step))}
        if c["train"]:
            s["gy"] = _randn(g, b, d, l, dtype=dt)
        return s
    b, l, d = c["batch"], c["seqlen"], c["dim"]
    # as AMADEUS forms them: decay exp(dt A) with A = -(1..64) over 6 heads
    dt_ = F.softplus(_randn(g, b, l, d, scale=0.5) - 4.0)
    a = -(torch.arange(d, device="cuda") % 64 + 1).float()
    s = {"dA": torch.exp(dt_ * a), "dBx": dt_ * _randn(g, b, l, d) * _randn(g, b, l, d), "C": _randn(g, b, l, d),
         "D": torch.ones(d, device="cuda"), "x": _randn(g, b, l, d)}
    if c["train"]:
        s["gy"] = _randn(g, b, l, d)
    return s


_LEAVES = {"add_rmsnorm_train": ("x", "r", "w"), "ce": ("x",), "lmhead": ("h", "w"),
           "scan": ("u", "delta", "A", "B", "C", "D", "z", "bias"), "diag": ("dA", "dBx", "C", "D", "x")}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case.get("train", True):
        for k in _LEAVES.get(case["op"], ()):
            s[k] = s[k].detach().requires_grad_()
    if case["op"] == "lmhead":
        from kernels.hip.chunked_linear_cross_entropy import ChunkedLinearCrossEntropyLoss
        s["loss_fn"] = ChunkedLinearCrossEntropyLoss(softcap=case["softcap"], label_smoothing=case["smoothing"])
    elif case["op"] in ("add_rmsnorm_train", "diag"):
        import kernels.hip._torch_ops  # noqa: F401  (registers torch.ops.autokernel)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def run(s):
    c = s["case"]
    op = c["op"]
    if op == "rmsnorm":
        from kernels.hip.rmsnorm import kernel_fn
        return kernel_fn(s["x"], s["w"])
    if op == "add_rmsnorm":
        from kernels.hip.fused_residual_add_rmsnorm import kernel_fn_dual
        return kernel_fn_dual(s["x"], s["r"], s["w"], eps=1e-5)
    if op == "add_rmsnorm_train":
        h, y = torch.ops.autokernel.fused_res_rmsnorm(s["x"], s["r"], s["w"], 1e-5)
        return (h.detach(), y.detach()) + torch.autograd.grad((h, y), (s["x"], s["r"], s["w"]), (s["gh"], s["gy"]))
    if op == "softmax":
        from kernels.hip.softmax import kernel_fn
        return kernel_fn(s["x"])
    if op == "ce":
        from kernels.ce_fused import ce_full
        loss = ce_full(s["x"], s["t"], softcap=c["softcap"], label_smoothing=c["smoothing"], mode=c["mode"],
                       z_loss_weight=c["z_loss"])
        return (loss.detach(),) + torch.autograd.grad(loss, s["x"])
    if op == "lmhead":
        if not c["train"]:
            with torch.no_grad():
                return s["loss_fn"](s["h"], s["w"], s["t"])
        loss = s["loss_fn"](s["h"], s["w"], s["t"])
        return (loss.detach(),) + torch.autograd.grad(loss, (s["h"], s["w"]))
    if op == "scan":
        from kernels.hip.selective_scan import selective_scan_fn
        args = (s["u"], s["delta"], s["A"], s["B"], s["C"], s["D"], s["z"], s["bias"], True)
        if not c["train"]:
            with torch.no_grad():
                return selective_scan_fn(*args, return_last_state=True)
        y = selective_scan_fn(*args)
        return (y.detach(),) + torch.autograd.grad(y, [s[k] for k in _LEAVES["scan"]], s["gy"])
    args = (s["dA"], s["dBx"], s["C"], s["D"], s["x"])
    if not c["train"]:
        with torch.no_grad():
            return torch.ops.autokernel.selective_scan(*args)
    y = torch.ops.autokernel.selective_scan(*args)
    return (y.detach(),) + torch.autograd.grad(y, args, s["gy"])


def work(case):
    c = case
    op, e = c["op"], _SIZE.get(c.get("dtype"), 4)
    if op in ("rmsnorm", "add_rmsnorm", "add_rmsnorm_train"):
        n = c["rows"] * c["cols"]
        # x, y | x, r, h, y | those, both output gradients and grad_x (grad_r is the same tensor)
        tensors = {"rmsnorm": 2, "add_rmsnorm": 4, "add_rmsnorm_train": 7}[op]
        return {"bytes": tensors * n * e, "flops": {"rmsnorm": 4, "add_rmsnorm": 5, "add_rmsnorm_train": 16}[op] * n}
    if op == "softmax":
        n = c["rows"] * c["cols"]
        return {"bytes": 2 * n * e, "flops": 5 * n}
    if op == "ce":
        n = c["rows"] * c["vocab"]
        return {"bytes": 2 * n * e + 8 * c["rows"], "flops": 8 * n}
    if op == "lmhead":
        m, v, d = c["rows"], c["vocab"], c["d"]
        # logits; in training also both gradient products, which need the
        # logits' softmax and so either their recomputation or their storage
        k = 3 if c["train"] else 1
        return {"bytes": (2 if c["train"] else 1) * (m + v) * d * e + 8 * m, "flops": k * 2 * m * v * d}
    if op == "scan":
        b, d, l, n = c["batch"], c["dim"], c["seqlen"], c["dstate"]
        wide, narrow = b * d * l, b * n * l
        if not c["train"]:  # u, delta, z, out; B, C; the last state
            return {"bytes": 4 * wide * e + 2 * narrow * e + 4 * b * d * n, "flops": 7 * wide * n}
        # and dout, du, ddelta, dz; dB, dC
        return {"bytes": 8 * wide * e + 4 * narrow * e, "flops": 21 * wide * n}
    n = c["batch"] * c["seqlen"] * c["dim"]
    # dA, dBx, C, x, y; and grad_y and the four gradients
    return {"bytes": (10 if c["train"] else 5) * n * 4, "flops": (14 if c["train"] else 4) * n}


def tolerance(case):
    op, dt = case["op"], case.get("dtype", "f32")
    if op == "lmhead" and not case["train"]:
        return {"rel": 1e-5, "max": 1e-5}  # the loss, a 32-bit sum
    if op == "ce" and dt == "f16":
        return {"rel": 2.2e-2, "max": 5e-2}  # small gradients round in fp16's subnormal range: 5.6e-3 off float64
    # outputs rounded once to their type, 2e-4 (fp16) and 1.7e-3 (bf16) off
    # float64; the scan's dz, from an output rounded to the type, 2.3e-3
    return {"f32": {"rel": 1e-5, "max": 1e-3}, "f16": {"rel": 1.2e-3, "max": 2e-2},
            "bf16": {"rel": 9e-3, "max": 1e-1}}[dt]


# ---------------------------------------------------------------------------
# The same in float64 torch
# ---------------------------------------------------------------------------

def _norm64(h, w, eps):
    return h * (h.square().mean(-1, keepdim=True) + eps).rsqrt() * w


def _ce64(x, t, softcap, smoothing, z_loss):
    if softcap > 0:
        x = softcap * torch.tanh(x / softcap)
    keep = t != -100
    lse = x.logsumexp(-1)
    xt = x.gather(1, t.clamp(min=0)[:, None])[:, 0]
    loss = lse - (1 - smoothing) * xt - smoothing * x.mean(-1) + z_loss * lse.square()
    return torch.where(keep, loss, 0.0).sum() / keep.sum().clamp(min=1)


def _scan64(s, case):
    l = case["seqlen"]
    u, z, B, C = (s[k].double() for k in ("u", "z", "B", "C"))
    A, D = s["A"].double(), s["D"].double()
    raw = s["delta"].double() + s["bias"].double()[:, None]
    delta = F.softplus(raw)
    # states before and after each step, time first
    n = case["dstate"]
    hs = torch.zeros(l + 1, case["batch"], case["dim"], n, dtype=torch.float64, device="cuda")
    y = torch.empty_like(u)
    dt, bt, ct, du_in = delta.permute(2, 0, 1), B.permute(2, 0, 1), C.permute(2, 0, 1), (delta * u).permute(2, 0, 1)
    for i in range(l):
        torch.addcmul(du_in[i][..., None] * bt[i][:, None], torch.exp(dt[i][..., None] * A), hs[i], out=hs[i + 1])
        y[..., i] = torch.einsum("bdn,bn->bd", hs[i + 1], ct[i])
    yd = y + D[:, None] * u
    gate = torch.sigmoid(z)
    out = yd * z * gate
    if not case["train"]:
        return out, hs[l].clone()
    go = s["gy"].double()
    dz = go * yd * gate * (1 + z * (1 - gate))
    dy = go * z * gate
    dyt, ut = dy.permute(2, 0, 1), u.permute(2, 0, 1)
    g = torch.zeros_like(hs[0])
    dA = torch.zeros_like(A)
    dB, dC, ddelta, du = torch.empty_like(B), torch.empty_like(C), torch.empty_like(u), torch.empty_like(u)
    for i in reversed(range(l)):
        g = g + dyt[i][..., None] * ct[i][:, None]
        dC[..., i] = torch.einsum("bd,bdn->bn", dyt[i], hs[i + 1])
        dB[..., i] = torch.einsum("bd,bdn->bn", du_in[i], g)
        gb = torch.einsum("bdn,bn->bd", g, bt[i])
        du[..., i] = dt[i] * gb
        g = g * torch.exp(dt[i][..., None] * A)
        w = g * hs[i]
        ddelta[..., i] = ut[i] * gb + (w * A).sum(-1)
        dA += (w * dt[i][..., None]).sum(0)
    ddelta = ddelta * torch.sigmoid(raw)
    return (out, du + D[:, None] * dy, ddelta, dA, dB, dC, (dy * u).sum((0, 2)), dz, ddelta.sum((0, 2)))


def _diag64(s, case):
    dA, dBx, C, x = (s[k].double() for k in ("dA", "dBx", "C", "x"))
    D = s["D"].double()
    hs = torch.zeros(case["batch"], case["seqlen"] + 1, case["dim"], dtype=torch.float64, device="cuda")
    for i in range(case["seqlen"]):
        hs[:, i + 1] = dA[:, i] * hs[:, i] + dBx[:, i]
    y = C * hs[:, 1:] + D * x
    if not case["train"]:
        return y
    gy = s["gy"].double()
    gB = torch.empty_like(dA)
    g = torch.zeros_like(dA[:, 0])
    for i in reversed(range(case["seqlen"])):
        g = g + gy[:, i] * C[:, i]
        gB[:, i] = g
        g = g * dA[:, i]
    return y, gB * hs[:, :-1], gB, gy * hs[:, 1:], (gy * x).sum((0, 1)), gy * D


def exact(case, seed):
    s = _inputs(case, seed)
    c, op = case, case["op"]
    with torch.no_grad():
        if op == "rmsnorm":
            return _norm64(s["x"].double(), s["w"].double(), 1e-6)
        if op == "add_rmsnorm":  # the norm takes the rounded sum, which is also the first output
            h = (s["x"].double() + s["r"].double()).to(s["x"].dtype).double()
            return h, _norm64(h, s["w"].double(), 1e-5)
        if op == "softmax":
            return torch.softmax(s["x"].double(), -1)
        if op == "scan":
            return _scan64(s, c)
        if op == "diag":
            return _diag64(s, c)
    if op == "add_rmsnorm_train":
        h = (s["x"].double() + s["r"].double()).to(s["x"].dtype).double().requires_grad_()
        w = s["w"].double().requires_grad_()
        y = _norm64(h, w, 1e-5)
        gh, gw = torch.autograd.grad(y, (h, w), s["gy"].double())
        gh = gh + s["gh"].double()
        return h.detach(), y.detach(), gh, gh, gw
    if op == "ce":
        x = s["x"].double().requires_grad_()
        loss = _ce64(x, s["t"], c["softcap"], c["smoothing"], c["z_loss"])
        return (loss.detach(),) + torch.autograd.grad(loss, x)
    h, w = s["h"].double().requires_grad_(), s["w"].double().requires_grad_()
    loss = _ce64(h @ w.t(), s["t"], c["softcap"], c["smoothing"], 0.0)
    if not c["train"]:
        return loss.detach()
    return (loss.detach(),) + torch.autograd.grad(loss, (h, w))
