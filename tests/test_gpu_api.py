"""GPU: the drop-in surfaces end to end -- torch.ops.autokernel.* with autograd and
autocast, and autokernel.optimize on a small pre-norm transformer (the
reference's test_tier2_parity.py / test_autokernel_autograd_safety.py
checks: rel 5e-3 forward, grads finite and non-zero on every parameter)."""

import pytest
import torch
import torch.nn as nn

from gpu_util import gpu, need_gpu, say

pytestmark = gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_ops_forward_backward(dtype):
    need_gpu()
    import kernels.hip._torch_ops  # noqa: F401
    g = torch.Generator().manual_seed(0)
    x0 = torch.randn(64, 512, generator=g)
    r0 = torch.randn(64, 512, generator=g)
    w0 = 1 + 0.1 * torch.randn(512, generator=g)
    gy = torch.randn(64, 512, generator=g)
    say("ops fwd/bwd", dtype)
    x = x0.to(dtype).to(DEV).requires_grad_()
    r = r0.to(dtype).to(DEV).requires_grad_()
    w = w0.to(dtype).to(DEV).requires_grad_()
    h, n = torch.ops.autokernel.fused_res_rmsnorm(x, r, w, 1e-6)
    (n.float() * gy.to(DEV)).sum().backward()
    xr = x0.to(dtype).double().requires_grad_()
    rr = r0.to(dtype).double().requires_grad_()
    wr = w0.to(dtype).double().requires_grad_()
    hr = xr + rr
    nr = hr / torch.sqrt(hr.pow(2).mean(-1, keepdim=True) + 1e-6) * wr
    (nr * gy.double()).sum().backward()
    tol = 1e-4 if dtype == torch.float32 else 2e-2
    for a, b in ((x.grad, xr.grad), (w.grad, wr.grad)):
        rel = float((a.double().cpu() - b).norm() / b.norm())
        assert rel < tol, rel
    # the plain RMSNorm op: values against the oracle, gradients against
    # float64 autograd of the reference formula
    from oracle import ops
    xa = x0.to(dtype).to(DEV).requires_grad_()
    wa = w0.to(dtype).to(DEV).requires_grad_()
    y = torch.ops.autokernel.rmsnorm(xa, wa, 1e-6)
    assert y.dtype == dtype and y.shape == xa.shape
    want = ops.rmsnorm_f32_ref(x0.to(dtype), w0.to(dtype), 1e-6)  # fp32, rounded once
    ytol = {torch.float32: 1e-5, torch.float16: 2e-3, torch.bfloat16: 1.6e-2}[dtype]  # about 1 ulp
    assert torch.allclose(y.detach().cpu().double(), want.double(), rtol=ytol, atol=ytol)
    (y.float() * gy.to(DEV)).sum().backward()
    xb = x0.to(dtype).double().requires_grad_()
    wb = w0.to(dtype).double().requires_grad_()
    yb = xb / torch.sqrt(xb.pow(2).mean(-1, keepdim=True) + 1e-6) * wb
    (yb * gy.double()).sum().backward()
    for a, b in ((xa.grad, xb.grad), (wa.grad, wb.grad)):
        rel = float((a.double().cpu() - b).norm() / b.norm())
        assert rel < tol, rel


def test_autocast_follows_dtype():
    need_gpu()
    import kernels.hip._torch_ops  # noqa: F401
    x = torch.randn(8, 256, device=DEV)
    w = torch.ones(256, device=DEV)
    say("autocast")
    for dt in (torch.float16, torch.bfloat16):
        with torch.autocast("cuda", dtype=dt):
            assert torch.ops.autokernel.rmsnorm(x, w).dtype == dt
            h, n = torch.ops.autokernel.fused_res_rmsnorm(x, x, w)
            assert h.dtype == dt and n.dtype == dt
    assert torch.ops.autokernel.rmsnorm(x, w).dtype == torch.float32


class RMSNorm(nn.Module):
    def __init__(self, d, eps=1e-6):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(d) + 0.05 * torch.randn(d))
        self.eps = eps

    def forward(self, x):
        xf = x.float()
        return (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.eps)).to(x.dtype) * self.weight


class Attn(nn.Module):
    def __init__(self, d):
        super().__init__()
        self.wq = nn.Linear(d, d, bias=False)

    def forward(self, x, freqs_cis):
        return self.wq(x)


class Block(nn.Module):
    def __init__(self, d):
        super().__init__()
        self.attention = Attn(d)
        self.attention_norm = RMSNorm(d)
        self.feed_forward = nn.Sequential(nn.Linear(d, 4 * d, bias=False), nn.SiLU(),
                                          nn.Linear(4 * d, d, bias=False))
        self.ffn_norm = RMSNorm(d)

    def forward(self, x, freqs_cis):
        h = x + self.attention(self.attention_norm(x), freqs_cis)
        return h + self.feed_forward(self.ffn_norm(h))


class TinyLM(nn.Module):
    def __init__(self, d=256, n=3, vocab=1000):
        super().__init__()
        self.emb = nn.Embedding(vocab, d)
        self.layers = nn.ModuleList([Block(d) for _ in range(n)])
        self.norm = RMSNorm(d)
        self.out = nn.Linear(d, vocab, bias=False)

    def forward(self, tok):
        x = self.emb(tok)
        for b in self.layers:
            x = b(x, None)
        return self.out(self.norm(x))


def test_optimize_training_step_bf16():
    need_gpu()
    import autokernel
    torch.manual_seed(0)
    model = TinyLM().to(DEV)
    tok = torch.randint(0, 1000, (4, 64), device=DEV)
    say("optimize tiny LM")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        ref = model(tok).float()
    model = autokernel.optimize(model, training=True)
    rep = autokernel.report(model)
    assert rep["patterns"]["fused_residual_rmsnorm"]["modules_replaced"] == 3
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = model(tok).float()
    rel = float((out - ref).norm() / ref.norm())
    assert rel < 3e-2, rel  # bf16 residual stream through 3 blocks vs the fp32 one
    loss = nn.functional.cross_entropy(out.view(-1, 1000), tok.view(-1))
    loss.backward()
    for name, p in model.named_parameters():
        assert p.grad is not None and torch.isfinite(p.grad).all() and p.grad.abs().sum() > 0, name


@pytest.mark.parametrize("form", ["layout", "type", "address"])
@pytest.mark.parametrize("op", ["rmsnorm", "add_rmsnorm", "diag", "scan", "ce_tiny", "lmhead"])
def test_backward_of_repacked_saved_tensors(op, form):
    """Saved-tensor hooks that hand back another layout (columns first), a
    wider type (which every value survives) or an odd address: the gradients are
    those without hooks, as the values that the backward reads are."""
    need_gpu()
    import kernels.hip._torch_ops  # noqa: F401
    from kernels.ce_fused import ce_full
    from kernels.hip.chunked_linear_cross_entropy import ChunkedLinearCrossEntropyLoss
    from kernels.hip.selective_scan import selective_scan_fn
    g = torch.Generator().manual_seed(5)

    def r(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g).to(dtype).to(DEV).requires_grad_()

    f32 = torch.float32
    t = torch.randint(0, 96, (40,), generator=g).to(DEV)
    if op == "rmsnorm":
        args, fn = (r(40, 96), r(96)), torch.ops.autokernel.rmsnorm
    elif op == "add_rmsnorm":
        args, fn = (r(40, 96), r(40, 96), r(96)), lambda *a: torch.ops.autokernel.fused_res_rmsnorm(*a)[1]
    elif op == "diag":
        args = tuple(r(2, 40, 32, dtype=f32) for _ in range(3)) + (r(32, dtype=f32), r(2, 40, 32, dtype=f32))
        fn = torch.ops.autokernel.selective_scan
    elif op == "scan":
        args = (r(2, 32, 40), r(2, 32, 40), r(32, 16, dtype=f32), r(2, 16, 40), r(2, 16, 40), r(32, dtype=f32),
                r(2, 32, 40), r(32, dtype=f32))

        def fn(u, delta, A, *rest):
            return selective_scan_fn(u, delta, -A.abs(), *rest, True)
    elif op == "ce_tiny":
        args, fn = (r(40, 96),), lambda x: ce_full(x, t, mode="tiny")
    else:
        args, fn = (r(40, 64), r(96, 64)), lambda h, w: ChunkedLinearCrossEntropyLoss()(h, w, t)

    def pack(v):
        if form == "layout":
            return v.transpose(0, 1).contiguous().transpose(0, 1) if v.dim() > 1 else v.clone()
        if form == "address":
            return torch.cat((v.new_zeros(1), v.reshape(-1)))[1:].view(v.shape)
        return v.to(f32) if v.is_floating_point() and v.dim() == 1 else v.to(torch.int32) if v.dtype == torch.long else v

    def grads(out):
        up = torch.ones_like(out)
        return torch.autograd.grad(out, args, up)

    say("repacked saved tensors", op, form)
    want = grads(fn(*args))
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda v: v):
        out = fn(*args)
    got = grads(out)
    for a, w, v in zip(args, want, got):
        assert v.dtype == a.dtype and torch.equal(w, v)


class _NoGradient(torch.autograd.Function):
    """Takes any tensors and hands back no gradient for them."""

    @staticmethod
    def forward(ctx, *xs):
        ctx.n = len(xs)
        return sum(x.float().sum() for x in xs)

    @staticmethod
    def backward(ctx, g):
        return (None,) * ctx.n


@pytest.mark.parametrize("form", ["plain", "transposed", "mixed"])
@pytest.mark.parametrize("op", ["rmsnorm", "add_rmsnorm", "diag"])
def test_ops_whose_consumer_gives_no_gradient(op, form):
    """Every input's gradient is zeros then, by each route: plain calls, and
    transposed and mixed-type ones, which the native host side leaves alone."""
    need_gpu()
    import kernels.hip._torch_ops  # noqa: F401
    k = torch.ops.autokernel
    wt = torch.float32 if form == "mixed" else torch.bfloat16
    if op == "diag":
        shapes, dts = [(2, 8, 16)] * 3 + [(16,), (2, 8, 16)], [torch.float32] * 5
        dts[3] = torch.bfloat16 if form == "mixed" else torch.float32
        fn = k.selective_scan
    elif op == "rmsnorm":
        shapes, dts, fn = [(40, 96), (96,)], [torch.bfloat16, wt], k.rmsnorm
    else:
        shapes, dts, fn = [(40, 96)] * 2 + [(96,)], [torch.bfloat16] * 2 + [wt], k.fused_res_rmsnorm
    leaves = [torch.randn(*s, device=DEV).to(dt) for s, dt in zip(shapes, dts)]
    if form == "transposed":
        leaves[0] = leaves[0].transpose(-1, -2).contiguous()
    leaves = [v.requires_grad_() for v in leaves]
    args = [leaves[0].transpose(-1, -2) if form == "transposed" else leaves[0]] + leaves[1:]
    say("no gradient from the consumer", op, form)
    out = fn(*args)
    loss = _NoGradient.apply(*(out if isinstance(out, (tuple, list)) else (out,)))
    for leaf, g in zip(leaves, torch.autograd.grad(loss, leaves)):
        assert g.shape == leaf.shape and g.dtype == leaf.dtype and not g.any()


def test_arguments_that_are_converted():
    """Numbers of another kind than the kernels' arguments, and limits beyond
    64 bits, are taken as the Python conversions take them."""
    need_gpu()
    from kernels.ce_fused import ce_full
    from kernels.hip import chunked_linear_cross_entropy as clc, selective_scan as ss
    g = torch.Generator().manual_seed(9)
    x, t = torch.randn(40, 96, generator=g).bfloat16().to(DEV), torch.randint(0, 96, (40,), generator=g).to(DEV)
    t[3] = -100
    say("converted arguments")
    want = ce_full(x, t, softcap=3.0, label_smoothing=0.5)
    assert torch.equal(ce_full(x, t, softcap="3", label_smoothing="0.5", ignore_index=-100.0), want)
    with pytest.raises(TypeError):
        ce_full(x, t, softcap=None)

    def lmhead():
        h, w = (torch.ones(40, 64, device=DEV, dtype=torch.bfloat16).requires_grad_() for _ in range(2))
        return torch.autograd.grad(clc.ChunkedLinearCrossEntropyLoss()(h, w, t % 40), (h, w))

    want = lmhead()
    for budget in (4e9, float("inf"), 1 << 70):
        with pytest.MonkeyPatch.context() as m:
            m.setattr(clc, "GRAD_LOGITS_BUDGET", budget)
            for a, b in zip(lmhead(), want):
                assert torch.equal(a, b)

    def kept(limit):  # bytes that a recorded scan holds beside its output
        ss.set_save_states(True, limit)
        try:
            u = torch.zeros(1, 64, 1024, device=DEV).requires_grad_()
            A, B = -torch.ones(64, 16, device=DEV), torch.zeros(1, 16, 1024, device=DEV)
            before = torch.cuda.memory_allocated()
            out = ss.selective_scan_fn(u, u, A, B, B)
            return torch.cuda.memory_allocated() - before - out.numel() * out.element_size()
        finally:
            ss.set_save_states(True, None)

    assert kept(-1) == kept(0) == 0
    assert kept(None) == kept(1 << 70) == kept(4 * 64 * 64 * 16) > 0 == kept(4 * 64 * 64 * 16 - 1)


def test_tensor_subclasses_keep_their_route():
    """A tensor subclass (no dispatch of its own) comes back as one where the
    result is made like the input, as torch makes it."""
    need_gpu()
    from kernels.hip.rmsnorm import kernel_fn as rmsnorm
    from kernels.hip.selective_scan import kernel_fn as diag

    class Tagged(torch.Tensor):
        pass

    x, w = torch.randn(8, 64, device=DEV), torch.randn(64, device=DEV)
    v = [torch.rand(2, 8, 16, device=DEV) for _ in range(4)]
    D = torch.rand(16, device=DEV)
    say("tensor subclasses")
    y = rmsnorm(x.as_subclass(Tagged), w)
    s = diag(v[0].as_subclass(Tagged), v[1], v[2], D, v[3])
    assert type(y) is Tagged and type(s) is Tagged
    assert torch.equal(y.as_subclass(torch.Tensor), rmsnorm(x, w))
    assert torch.equal(s.as_subclass(torch.Tensor), diag(*v[:3], D, v[3]))
    assert type(rmsnorm(x, torch.nn.Parameter(w))) is torch.Tensor


def test_function_modes_and_the_native_route(monkeypatch):
    """A default device does not keep calls from the native side; a function mode
    that looks at torch's calls sees them, from the Python form."""
    need_gpu()
    from torch.overrides import TorchFunctionMode
    from kernels.hip import _lib
    from kernels.hip.softmax import kernel_fn as softmax

    class Watch(TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.seen = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.seen.append(getattr(func, "__name__", ""))
            return func(*args, **(kwargs or {}))

    say("function modes")
    x = torch.randn(4, 64, device=DEV)
    want = softmax(x)
    python = []
    launch = _lib.softmax
    monkeypatch.setattr(_lib, "softmax", lambda *a: python.append(1) or launch(*a))
    with torch.device(DEV):
        assert _lib.native(x) is not None and torch.equal(softmax(x), want)
    with torch.device("cpu"):
        y = softmax(x)
    assert y.is_cuda and torch.equal(y, want) and not python
    with Watch() as w, torch.device(DEV):
        y = softmax(x)
    assert torch.equal(y, want) and python and "empty" in w.seen


def test_rows_of_no_columns():
    need_gpu()
    from kernels.hip.rmsnorm import kernel_fn as rmsnorm
    say("rows of no columns")
    assert rmsnorm(torch.empty(4, 0, device=DEV), torch.empty(0, device=DEV)).shape == (4, 0)


@pytest.mark.parametrize("op", ["rmsnorm", "add_rmsnorm", "diag", "scan", "scan_last", "ce", "ce_tiny", "lmhead"])
def test_compiled_autograd(op):
    """A backward that torch's compiled autograd records gives the eager one's bits."""
    need_gpu()
    import kernels.hip._torch_ops  # noqa: F401
    import torch._dynamo.compiled_autograd as compiled
    from kernels.ce_fused import ce_full
    from kernels.hip.chunked_linear_cross_entropy import ChunkedLinearCrossEntropyLoss
    from kernels.hip.selective_scan import selective_scan_fn
    g = torch.Generator().manual_seed(6)
    t = torch.randint(0, 96, (40,), generator=g).to(DEV)

    def r(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g).to(dtype).to(DEV).requires_grad_()

    f32 = torch.float32
    if op == "rmsnorm":
        args, fn = (r(40, 96), r(96)), torch.ops.autokernel.rmsnorm
    elif op == "add_rmsnorm":
        args, fn = (r(40, 96), r(40, 96), r(96)), lambda *a: torch.ops.autokernel.fused_res_rmsnorm(*a)[1]
    elif op == "diag":
        args = tuple(r(2, 40, 32, dtype=f32) for _ in range(3)) + (r(32, dtype=f32), r(2, 40, 32, dtype=f32))
        fn = torch.ops.autokernel.selective_scan
    elif op.startswith("scan"):
        args = (r(2, 32, 40), r(2, 32, 40), r(32, 16, dtype=f32), r(2, 16, 40), r(2, 16, 40), r(32, dtype=f32),
                r(2, 32, 40), r(32, dtype=f32))

        def fn(u, delta, A, *rest):
            y = selective_scan_fn(u, delta, -A.abs(), *rest, True, op == "scan_last")
            return y[0] if op == "scan_last" else y
    elif op.startswith("ce"):
        args, fn = (r(40, 96),), lambda x: ce_full(x, t, mode="tiny" if op == "ce_tiny" else "fused")
    else:
        args, fn = (r(40, 64), r(96, 64)), lambda h, w: ChunkedLinearCrossEntropyLoss()(h, w, t)
    say("compiled autograd", op)
    want = torch.autograd.grad(fn(*args).sum(), args)
    loss = fn(*args).sum()
    with compiled._enable(torch.compile(backend="eager")):
        loss.backward()
    for a, w in zip(args, want):
        assert torch.equal(a.grad, w)


def _entry_point(name, g):
    """(leaves, function of them to one or several outputs) of an entry point."""
    from kernels import ce_fused
    from kernels.hip import fused_residual_add_rmsnorm as add, rmsnorm, selective_scan as ss, softmax
    from kernels.hip.chunked_linear_cross_entropy import ChunkedLinearCrossEntropyLoss
    f32, k = torch.float32, torch.ops.autokernel

    def r(*shape, dtype=torch.bfloat16):
        return torch.randn(*shape, generator=g).to(dtype).to(DEV).requires_grad_()

    t = torch.randint(0, 96, (40,), generator=g).to(DEV)
    t[7] = -100
    norm = (r(40, 96), r(96))
    add_norm = (r(40, 96), r(40, 96), r(96))
    diag = tuple(r(2, 40, 32, dtype=f32) for _ in range(3)) + (r(32, dtype=f32), r(2, 40, 32, dtype=f32))
    scan = (r(2, 32, 70), r(2, 32, 70), r(32, 16, dtype=f32), r(2, 16, 70), r(2, 16, 70), r(32, dtype=f32), r(2, 32, 70),
            r(32, dtype=f32))

    def mamba(last):
        return lambda u, d, A, *rest: ss.selective_scan_fn(u, d, -A.abs(), *rest, True, last)

    def plain(fn):  # no gradient: outputs alone
        def call(*a):
            with torch.no_grad():
                return fn(*a)
        return call

    return {
        "rmsnorm": (norm, plain(rmsnorm.kernel_fn)), "add_rmsnorm": (add_norm, plain(add.kernel_fn)),
        "add_rmsnorm_dual": (add_norm, plain(add.kernel_fn_dual)), "softmax": (norm[:1], plain(softmax.kernel_fn)),
        "diag": (diag, plain(ss.kernel_fn)), "rmsnorm_op": (norm, k.rmsnorm), "add_rmsnorm_op": (add_norm, k.fused_res_rmsnorm),
        "diag_op": (diag, k.selective_scan), "scan": (scan, mamba(False)), "scan_last": (scan, mamba(True)),
        "ce": (norm[:1], lambda x: ce_fused.kernel_fn(x, t)),
        "ce_fused": (norm[:1], lambda x: ce_fused.ce_full(x, t, softcap=5.0, z_loss_weight=1e-3, return_z=True)),
        "ce_tiny": (norm[:1], lambda x: ce_fused.ce_full(x, t, mode="tiny", label_smoothing=0.1)),
        "lmhead": ((r(40, 64), r(96, 64)), lambda h, w: ChunkedLinearCrossEntropyLoss(softcap=5.0)(h, w, t)),
    }[name]


@pytest.mark.parametrize("name", ["rmsnorm", "add_rmsnorm", "add_rmsnorm_dual", "softmax", "diag", "rmsnorm_op", "add_rmsnorm_op",
                                  "diag_op", "scan", "scan_last", "ce", "ce_fused", "ce_tiny", "lmhead"])
def test_native_and_python_routes_agree(name, monkeypatch):
    """Every entry point with the native host side and with it switched off (the
    form that takes converted, wrapped and traced calls): the same kernels, so the
    same bits of every output and gradient."""
    need_gpu()
    import kernels.hip._torch_ops  # noqa: F401
    from kernels.hip import _lib
    leaves, fn = _entry_point(name, torch.Generator().manual_seed(12))

    def run():
        out = fn(*leaves)
        out = out if isinstance(out, (tuple, list)) else (out,)
        diff = [o for o in out if o.requires_grad]
        return [o.detach() for o in out] + list(torch.autograd.grad(diff, leaves, [torch.full_like(o, 0.5) for o in diff]) if diff else [])

    say("native and python routes", name)
    native = run()
    used = []
    monkeypatch.setattr(_lib, "native", lambda *a: used.append(1))
    python = run()
    assert used and len(native) == len(python)
    for a, b in zip(native, python):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("op", ["rmsnorm_op", "add_rmsnorm_op", "diag_op"])
def test_formula_backwards_of_native_graphs(op, monkeypatch):
    """Graphs that the native side recorded before the backward kernels were
    switched off take the torch formulas, as graphs recorded after it do; both
    are the kernels' gradients within two roundings of the type (fp32: 1e-4 of
    the largest, over 40-step products)."""
    need_gpu()
    import kernels.hip._torch_ops as ops_module
    from kernels.hip import _lib
    leaves, fn = _entry_point(op, torch.Generator().manual_seed(13))

    def record():
        out = fn(*leaves)
        return out if isinstance(out, (tuple, list)) else (out,)

    def grads(out):
        return torch.autograd.grad(out, leaves, [torch.full_like(o, 0.5) for o in out])

    say("formula backwards", op)
    want = grads(record())
    recorded = record()
    monkeypatch.setattr(ops_module, "_BWD_KERNELS_ENABLED", True)  # restored at the end
    ops_module.disable_hip_backward()
    try:
        before, after = grads(recorded), grads(record())
    finally:
        _lib.host().set_hip_backward(True)
    unit = 2.0 ** -7 if leaves[0].dtype == torch.bfloat16 else 1e-4
    for w, a, b in zip(want, before, after):
        assert a.dtype == b.dtype == w.dtype and torch.equal(a, b)
        assert bool(((a.double() - w.double()).abs() <= 2 * unit * w.double().abs() + unit * 0.1 * w.double().abs().amax()).all())
