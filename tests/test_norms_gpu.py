"""The fused normalisations against float64 torch (GPU), at the edges of the
lane layouts (rows of up to 128, 768, 2048 and 4096 elements) and of a
workgroup's rows, and the calls that stay on the torch expressions."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from representax_amd import norms, ops
from representax_amd.norms import LayerNorm, RMSNorm, add_norm, attention_heads

DEV = "cuda:0"
BF16, F64 = torch.bfloat16, torch.float64
# one rounding to bf16 moves a value by at most 2^-9 of itself; f32 sums of at
# most 4096 terms and the f32 reciprocal root are far below a quarter of that
ONE_ROUNDING = 1.25 * 2.0 ** -9


def _rel(a, b):
    return float((a.to(F64) - b).norm() / b.norm().clamp_min(1e-300))


def _module(kind, size, device=DEV, seed=0):
    g = torch.Generator().manual_seed(seed)
    norm = LayerNorm(size, 1e-12, device) if kind == "layer" else RMSNorm(size, 1e-6, device)
    with torch.no_grad():
        for p in norm.parameters():
            p.copy_(1.0 + 0.5 * torch.randn(size, generator=g))
    return norm.requires_grad_(False)


def _want(norm, t):
    """The norm in float64; the LayerNorm takes its weights in bf16."""

    if isinstance(norm, LayerNorm):
        w, b = (p.to(BF16).to(F64) for p in (norm.weight, norm.bias))
        return F.layer_norm(t, t.shape[-1:], w, b, norm.eps)
    return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + norm.eps) * norm.weight.to(F64)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["layer", "rms"])
@pytest.mark.parametrize("rows,size", [(1, 8), (33, 128), (17, 136), (9, 768), (7, 776),
                                       (5, 2048), (3, 2056), (2, 4096)])
def test_norm_and_residual_norm(kind, rows, size):
    g = torch.Generator().manual_seed(rows * size)
    x, r, dy, dt = (torch.randn(rows, size, generator=g).to(DEV, BF16) for _ in range(4))
    norm = _module(kind, size)
    x.requires_grad_(True)
    r.requires_grad_(True)
    y = norm(x)
    assert "NormFn" in type(y.grad_fn).__name__
    x64 = x.detach().to(F64).requires_grad_(True)
    want = _want(norm, x64)
    assert _rel(y, want) <= ONE_ROUNDING
    (dx,) = torch.autograd.grad(y, x, dy)
    (dx64,) = torch.autograd.grad(want, x64, dy.to(F64))
    # a row of 8 under the LayerNorm keeps little of its gradient (two of its
    # eight directions are projected out), still one rounding of what is left
    assert _rel(dx, dx64) <= ONE_ROUNDING

    t, y = add_norm(norm, x, r)
    assert torch.equal(t, x + r)
    t64 = t.detach().to(F64).requires_grad_(True)
    want = _want(norm, t64)
    assert _rel(y, want) <= ONE_ROUNDING
    dx, dr = torch.autograd.grad([t, y], [x, r], [dt, dy], retain_graph=True)
    (d64,) = torch.autograd.grad(want, t64, dy.to(F64), retain_graph=True)
    assert torch.equal(dx, dr)
    assert _rel(dx, d64 + dt.to(F64)) <= ONE_ROUNDING
    # either output alone, the gradient of the norm as a transposed view
    (only,) = torch.autograd.grad(t, x, dt, retain_graph=True)
    assert torch.equal(only, dt)
    (only,) = torch.autograd.grad(y, x, dy.t().contiguous().t())
    assert _rel(only, d64) <= ONE_ROUNDING


@pytest.mark.gpu
@pytest.mark.parametrize("b,s,h,d,repeat", [(1, 1, 1, 64, 1), (2, 5, 3, 128, 2), (1, 17, 8, 64, 3),
                                            (3, 7, 16, 128, 1)])
@pytest.mark.parametrize("weight_dtype", [torch.float32, BF16])
def test_head_norm_with_rotation(b, s, h, d, repeat, weight_dtype):
    g = torch.Generator().manual_seed(b * s * h)
    x = torch.randn(b, s, h, d, generator=g).to(DEV, BF16).requires_grad_(True)
    angle = torch.randn(1, s, d // 2, generator=g).repeat(1, 1, 2).to(DEV)
    cos, sin = angle.cos(), angle.sin()
    norm = _module("rms", d).to(weight_dtype)
    # queries of h * repeat heads beside keys and values of h heads
    q = torch.randn(b, s, h * repeat, d, generator=g).to(DEV, BF16).requires_grad_(True)
    v = torch.randn(b, s, h, d, generator=g).to(DEV, BF16).requires_grad_(True)
    query_norm = _module("rms", d, seed=1).to(weight_dtype)
    outs = attention_heads(query_norm, norm, q, x, v, cos, sin, BF16)
    assert "HeadNormFn" in type(outs[1].grad_fn).__name__
    dy = torch.randn(b, h * repeat, s, d, generator=g).to(DEV, BF16).transpose(1, 2)
    for n, t, y, rep in ((query_norm, q, outs[0], 1), (norm, x, outs[1], repeat)):
        t64 = t.detach().to(F64).requires_grad_(True)
        n64 = _want(n, t64)
        half = torch.cat((-n64[..., d // 2:], n64[..., :d // 2]), dim=-1)
        want = (n64 * cos.to(F64)[:, :, None] + half * sin.to(F64)[:, :, None])
        want = want.repeat_interleave(rep, dim=2)
        # the normalised value rounds, the rotation keeps its length, the sum rounds
        assert _rel(y, want) <= 2 * ONE_ROUNDING
        (dx,) = torch.autograd.grad(y, t, dy, retain_graph=True)
        (dx64,) = torch.autograd.grad(want, t64, dy.to(F64))
        assert _rel(dx, dx64) <= ONE_ROUNDING
        (again,) = torch.autograd.grad(y, t, dy.contiguous(), retain_graph=True)
        assert torch.equal(dx, again)
    assert torch.equal(outs[2], v.repeat_interleave(repeat, dim=2))
    (dv,) = torch.autograd.grad(outs[2], v, dy, retain_graph=True)
    assert _rel(dv, dy.to(F64).reshape(b, s, h, repeat, d).sum(3)) <= ONE_ROUNDING
    # all three at once
    found = torch.autograd.grad(outs, [q, x, v], [dy] * 3)
    assert torch.equal(found[1], dx) and torch.equal(found[2], dv)


@pytest.mark.gpu
def test_second_derivatives_and_torch_routes():
    x = torch.randn(4, 64, device=DEV).to(BF16).requires_grad_(True)
    r = torch.randn(4, 64, device=DEV).to(BF16)
    norm = _module("rms", 64)
    _, y = add_norm(norm, x, r)
    (dx,) = torch.autograd.grad(y.float().square().sum(), x, create_graph=True)
    (ddx,) = torch.autograd.grad(dx.float().square().sum(), x)
    want = x.detach().to(F64).requires_grad_(True)
    t = (x + r).detach().to(F64) - x.detach().to(F64)
    (d1,) = torch.autograd.grad(_want(norm, want + t).square().sum(), want, create_graph=True)
    (d2,) = torch.autograd.grad(d1.square().sum(), want)
    # intermediate bf16 gradients (a handful of roundings, partly cancelling)
    assert _rel(ddx, d2) <= 16 * ONE_ROUNDING

    # weights that want a gradient, hooks, autocast, transforms, layouts
    assert norms._row_kernel(x, norm.weight)
    assert not norms._row_kernel(x.t(), norm.weight) and not norms._row_kernel(x[:, :60], norm.weight)
    norm.weight.requires_grad_(True)
    add_norm(norm, x, r)[1].sum().backward()
    assert norm.weight.grad is not None
    with torch.no_grad():
        assert norms._row_kernel(x, norm.weight)
    norm.weight.requires_grad_(False)
    seen = []
    handle = norm.register_forward_hook(lambda m, a, out: seen.append(a[0]))
    t, _ = add_norm(norm, x, r)
    assert seen and torch.equal(seen[0], t)
    handle.remove()
    with torch.autocast("cuda", dtype=BF16):
        assert not norms._row_kernel(x, norm.weight)
    rows = torch.func.vmap(norm)(x.detach())
    assert _rel(rows, _want(norm, x.detach().to(F64))) <= 2 * ONE_ROUNDING
    _, tangent = torch.func.jvp(lambda v: norm(v), (x.detach(),), (r,))
    assert torch.isfinite(tangent).all()


def test_expressions_on_the_cpu():
    x, r = torch.randn(3, 16), torch.randn(3, 16)
    for kind in ("layer", "rms"):
        norm = _module(kind, 16, "cpu")
        t, y = add_norm(norm, x, r)
        assert torch.equal(t, x + r) and torch.equal(y, norm(x + r))
    q, k, v = (torch.randn(2, 5, n, 64) for n in (6, 3, 3))
    angle = torch.randn(1, 5, 32).repeat(1, 1, 2)
    norm = _module("rms", 64, "cpu")
    got = attention_heads(norm, norm, q, k, v, angle.cos(), angle.sin(), torch.float32)
    turned = [norms.rotate(norm(t), angle.cos(), angle.sin()) for t in (q, k)]
    assert torch.equal(got[0], turned[0])
    assert torch.equal(got[1], turned[1].repeat_interleave(2, dim=2))
    assert torch.equal(got[2], v.repeat_interleave(2, dim=2))


@pytest.mark.parametrize("kv,route", [((2, 5, 2, 64), True), ((2, 5, 4, 64), True),
                                      ((2, 3, 2, 64), False), ((1, 5, 2, 64), False),
                                      ((2, 5, 2, 128), False), ((2, 5, 3, 64), False)])
def test_attention_heads_launches_only_over_matching_tokens(monkeypatch, kv, route):
    """The launch reads the queries' token count of every part: keys and values
    of other tokens, batches or head widths (or head counts that do not divide
    the queries') stay on the torch expressions, which raise or broadcast."""

    taken = []
    monkeypatch.setattr(norms, "plain_tensor", lambda t: True)
    monkeypatch.setattr(norms, "_rows_fit", lambda *a: True)
    monkeypatch.setattr(RMSNorm, "forward", lambda m, t: norms.rms_norm(t, m.weight, m.eps))
    monkeypatch.setattr(norms.HeadNormFn, "apply", lambda *a: taken.append(a) or (q, k, v))
    q, k, v = (torch.randn(s).to(BF16) for s in ((2, 5, 4, 64), kv, kv))
    norm, key_norm = _module("rms", 64, "cpu"), _module("rms", kv[3], "cpu")
    angle = torch.randn(1, 5, 32).repeat(1, 1, 2)
    call = (norm, key_norm, q, k, v, angle.cos(), angle.sin(), BF16)
    if kv[1] != 5 or kv[3] != 64:
        with pytest.raises(RuntimeError):  # the rotation meets angles of other tokens
            attention_heads(*call)
    else:
        outs = attention_heads(*call)
        if kv[0] == 1:  # a batch that attention broadcasts
            assert outs[1].shape == outs[2].shape == (1, 5, 4, 64)
    assert bool(taken) == route
    if not route and kv[2] == 2:
        with pytest.raises(ValueError, match="same tokens"):
            norms._head_norm(angle, angle, ((1e-6, 1),) * 2, (q, k), (norm.weight,) * 2, None, None)


def _cpu_routes(monkeypatch):
    """The routes' conditions on CPU tensors: everything but their device."""

    def plain(t):
        return type(t) in (torch.Tensor, torch.nn.Parameter) and torch._C._has_storage(t)

    monkeypatch.setattr(norms, "plain_tensor", plain)
    monkeypatch.setattr(norms, "on_current_device", lambda t: True)


def test_transforms_and_compilers_keep_the_expressions(monkeypatch):
    """Inside a function transform a tensor that is closed over is no wrapper,
    but an autograd function is refused all the same; a compiler cannot trace
    the conditions. Both get the torch expressions."""

    _cpu_routes(monkeypatch)
    x, r = (torch.randn(4, 16).to(BF16) for _ in range(2))
    norm, bias = _module("rms", 16, "cpu"), _module("layer", 16, "cpu")
    assert norms._row_kernel(x, norm.weight)
    seen = []

    def closed_over(value):
        seen.append(norms._row_kernel(x, norm.weight))
        return add_norm(norm, x, r)[1].float().sum() * value

    torch.func.vmap(closed_over)(torch.ones(3))
    torch.func.grad(closed_over)(torch.ones(()))
    torch.func.jvp(closed_over, (torch.ones(()),), (torch.ones(()),))
    assert seen == [False] * 3
    for module in (norm, bias):
        compiled = torch.compile(module, fullgraph=True, backend="eager")
        assert torch.equal(compiled(x), norms._expression(
            int(module is norm), x, module.weight, getattr(module, "bias", None), module.eps))
    compiled = torch.compile(lambda v: add_norm(norm, v, r), fullgraph=True, backend="eager")
    assert torch.equal(compiled(x)[1], norms.rms_norm(x + r, norm.weight, norm.eps))
    angle = torch.randn(1, 5, 32).repeat(1, 1, 2)
    q, k, v = (torch.randn(2, 5, n, 64).to(BF16) for n in (4, 2, 2))
    head = _module("rms", 64, "cpu")
    compiled = torch.compile(lambda *t: attention_heads(head, head, *t, angle.cos(), angle.sin(), BF16),
                             fullgraph=True, backend="eager")
    assert torch.equal(compiled(q, k, v)[2], v.repeat_interleave(2, dim=2))


@pytest.mark.gpu
def test_transforms_and_compilers_on_the_device():
    x, r = (torch.randn(4, 64, device=DEV).to(BF16) for _ in range(2))
    norm = _module("rms", 64)
    want = norms.rms_norm(x + r, norm.weight, norm.eps)
    rows = torch.func.vmap(lambda c: add_norm(norm, x, r)[1] * c)(torch.ones(2, device=DEV, dtype=BF16))
    assert torch.equal(rows[1], want)
    compiled = torch.compile(lambda v: add_norm(norm, v, r)[1], fullgraph=True, backend="eager")
    assert torch.equal(compiled(x), want)
    masters = [torch.randn(8, 64, device=DEV) for _ in range(2)]
    views = torch.func.vmap(lambda c: ops.cast_many(masters, BF16)[0] * c)(
        torch.ones(2, device=DEV, dtype=BF16))
    assert torch.equal(views[0], masters[0].to(BF16))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["layer", "rms"])
def test_more_rows_than_one_grid_dimension(kind):
    """2^28 rows of 8 elements are 2^32 lanes, one more than a launch holds in a
    dimension: the rows on both sides of the limit equal the same rows' norms
    in a small call, forward and backward."""

    rows = (1 << 28) + 5
    g = torch.Generator(device=DEV).manual_seed(1)
    base, grad = (torch.randn(1 << 14, 8, generator=g, device=DEV).to(BF16) for _ in range(2))
    x, dy = (t.repeat(1 << 14, 1)[:rows] for t in (base, grad))
    x = torch.cat((x, base[:5]))[:rows].requires_grad_(True)
    dy = torch.cat((dy, grad[:5]))[:rows]
    norm = _module(kind, 8)
    y = norm(x)
    assert "NormFn" in type(y.grad_fn).__name__
    (dx,) = torch.autograd.grad(y, x, dy)
    small = base.clone().requires_grad_(True)
    want = norm(small)
    (dwant,) = torch.autograd.grad(want, small, grad)
    for got, part in ((y.detach(), want.detach()), (dx, dwant)):
        for at in (0, 1 << 25, (1 << 28) - (1 << 14)):  # row 0, the second grid row, the last
            assert torch.equal(got[at:at + (1 << 14)], part)
        assert torch.equal(got[1 << 28:], part[:5])
    del x, y, dx, dy, got
    torch.cuda.empty_cache()


@pytest.mark.gpu
def test_more_heads_than_one_grid_row():
    """2^21 workgroups of 32 heads and a few more: the second row of the grid."""

    s, h, d = (1 << 19) + 8, 128, 64
    g = torch.Generator(device=DEV).manual_seed(2)
    q = torch.randn(1, 64, h, d, generator=g, device=DEV).to(BF16)
    k, v = (torch.randn(1, 64, 1, d, generator=g, device=DEV).to(BF16) for _ in range(2))
    angle = torch.randn(1, 64, d // 2, generator=g, device=DEV).repeat(1, 1, 2)
    norm = _module("rms", d)
    want = attention_heads(norm, norm, q, k, v, angle.cos(), angle.sin(), BF16)

    def many(t):
        return t.repeat(1, -(-s // 64), *([1] * (t.dim() - 2)))[:, :s].contiguous()

    got = attention_heads(norm, norm, many(q), many(k), many(v), many(angle.cos()),
                          many(angle.sin()), BF16)
    for a, b in zip(got, want):
        for at in (0, 1 << 18, s - 8 - 64):
            assert torch.equal(a[:, at:at + 64], b)
        assert torch.equal(a[:, s - 8:], b[:, :8])
    del got, a
    torch.cuda.empty_cache()


@pytest.mark.gpu
def test_the_argument_of_an_rms_norm_may_change_before_the_backward():
    """The expression saves a float32 copy of a bf16 row, so changing the row in
    place after the call (x += ..., an RMSNorm's usual neighbour) is allowed.
    The LayerNorm's expression saves its argument, where it is not."""

    leaf = torch.randn(5, 64, device=DEV).to(BF16).requires_grad_(True)
    dy = torch.randn(5, 64, device=DEV).to(BF16)
    norm = _module("rms", 64)
    got = []
    for change in (False, True):
        x = leaf * 1.0
        y = norm(x)
        assert "NormFn" in type(y.grad_fn).__name__
        if change:
            x.add_(1.0)
        got.append((y.detach().clone(), *torch.autograd.grad(y, leaf, dy)))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    x = leaf * 1.0
    y = norm(x)
    (dx,) = torch.autograd.grad(y.float().square().sum(), x, create_graph=True)
    assert torch.autograd.grad(dx.float().sum(), leaf)[0].shape == leaf.shape


@pytest.mark.gpu
def test_tensors_of_another_device_than_the_current_one(monkeypatch):
    """A launch goes to the current device; torch's operations go to their
    tensors' device. Where the two differ the expressions run."""

    x, r = (torch.randn(4, 64, device=DEV).to(BF16) for _ in range(2))
    norm, masters = _module("rms", 64), [torch.randn(8, 8, device=DEV) for _ in range(2)]
    want = norms.rms_norm(x + r, norm.weight, norm.eps)
    assert norms._row_kernel(x, norm.weight)
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: 1)
    assert not norms._row_kernel(x, norm.weight)

    def no_launch(*args):
        raise AssertionError(args[0])

    monkeypatch.setattr(norms.nat, "call", no_launch)
    assert torch.equal(add_norm(norm, x, r)[1], want) and torch.equal(norm(x + r), want)
    for t, got in zip(masters, ops.cast_many(masters, BF16)):
        assert torch.equal(got, t.to(BF16))


@pytest.mark.gpu
def test_heads_that_are_only_repeated_are_not_kept():
    q, k, v = (torch.randn(1, 3, n, 64, device=DEV).to(BF16).requires_grad_(True) for n in (4, 2, 2))
    angle = torch.randn(1, 3, 32, device=DEV).repeat(1, 1, 2)
    norm = _module("rms", 64)
    outs = attention_heads(norm, norm, q, k, v, angle.cos(), angle.sin(), BF16)
    kept = outs[2].grad_fn.saved_tensors
    assert len(kept) == 6 and not any(t is v for t in kept)
    (dv,) = torch.autograd.grad(outs[2], v, torch.ones_like(outs[2]), create_graph=True)
    assert torch.equal(dv, torch.full_like(v, 2.0))


@pytest.mark.gpu
@pytest.mark.parametrize("create_graph", [False, True])
def test_batched_gradients(create_graph):
    """Several gradients at once (is_grads_batched, vectorized Jacobians) have
    no storage for a kernel to read; the expressions are differentiated."""

    x, r = (torch.randn(3, 5, 64, device=DEV).to(BF16).requires_grad_(True) for _ in range(2))
    for kind in ("layer", "rms"):
        norm = _module(kind, 64)
        dy = torch.randn(4, 3, 5, 64, device=DEV).to(BF16)
        for y, leaves in ((norm(x), [x]), (add_norm(norm, x, r)[1], [x, r])):
            assert "NormFn" in type(y.grad_fn).__name__
            one = [torch.autograd.grad(y, leaves, g, retain_graph=True) for g in dy]
            all_ = torch.autograd.grad(y, leaves, dy, is_grads_batched=True, retain_graph=True,
                                       create_graph=create_graph)
            for i, got in enumerate(all_):
                assert got.shape == dy.shape
                for j in range(4):  # both within one rounding of float64
                    assert _rel(got[j], one[j][i].to(F64)) <= 2 * ONE_ROUNDING
    q, k, v = (torch.randn(2, 5, n, 64, device=DEV).to(BF16).requires_grad_(True) for n in (4, 2, 2))
    angle = torch.randn(1, 5, 32, device=DEV).repeat(1, 1, 2)
    norm = _module("rms", 64)
    outs = attention_heads(norm, norm, q, k, v, angle.cos(), angle.sin(), BF16)
    assert "HeadNormFn" in type(outs[1].grad_fn).__name__
    dy = torch.randn(3, 2, 5, 4, 64, device=DEV).to(BF16)
    for y, t in zip(outs, (q, k, v)):
        (got,) = torch.autograd.grad(y, t, dy, is_grads_batched=True, retain_graph=True,
                                     create_graph=create_graph)
        for j in range(3):
            (one,) = torch.autograd.grad(y, t, dy[j], retain_graph=True)
            # the expression rounds the rotated gradient, the repeated heads'
            # sum and the result, the kernel the result
            assert _rel(got[j], one.to(F64)) <= 4 * ONE_ROUNDING


def test_batched_gradients_reach_no_kernel(monkeypatch):
    _cpu_routes(monkeypatch)
    monkeypatch.setattr(norms, "_forward", lambda x, r, w, b, kind, eps: (
        None, norms._expression(kind, x, w, b, eps)))
    x = torch.randn(4, 16, dtype=torch.float32).to(BF16).requires_grad_(True)
    norm = _module("rms", 16, "cpu")
    y = norms.NormFn.apply(x, norm.weight, None, norms.nat.NORM_RMS, norm.eps)
    dy = torch.randn(5, 4, 16).to(BF16)
    with pytest.raises(RuntimeError, match="ROCm devices only"):  # one gradient: the kernel's
        torch.autograd.grad(y, x, dy[0], retain_graph=True)
    (got,) = torch.autograd.grad(y, x, dy, is_grads_batched=True)
    for i in range(5):
        (want,) = torch.autograd.grad(norms.rms_norm(x, norm.weight, norm.eps), x, dy[i])
        assert _rel(got[i], want.to(F64)) <= 2 * ONE_ROUNDING
