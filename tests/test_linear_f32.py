"""float32 linear layer and gradients on split fp16 operands (rpfq_linear_f32,
rpfq_linear_f32_grad) against float64.

Bar, per output: two 22-bit operands and the dropped low x low product cost
at most 2^-20 of sum |a| |b|, each of the 3 K / 16 float32 accumulations of
an output at most 2^-23 of it (the partial sums a matrix instruction rounds),
and values below 2^-39 of their row's largest (gw: of the tensor's) are lost.
"""
import ctypes

import numpy as np
import pytest
import torch

DEV = "cuda"


def _bound(a, b, con, floor):
    return (2.0 ** -20 + 3 * (con / 16 + 1) * 2.0 ** -23) * (a.abs() @ b.abs()) + floor


def _inputs(m, n, k, seed=0, dev=DEV):
    g = torch.Generator(device=dev).manual_seed(seed)
    x = torch.randn(m, k, device=dev, generator=g)
    x *= torch.exp2(torch.randint(-3, 4, (m, 1), device=dev, generator=g).float())
    w = torch.randn(n, k, device=dev, generator=g) * 0.02
    gy = torch.randn(m, n, device=dev, generator=g) * 1e-3
    return x, w, torch.randn(n, device=dev, generator=g), gy


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (15, 40, 24), (16, 256, 32), (65, 264, 40), (96, 128, 64), (127, 8, 776),
                                   (129, 1000, 264), (385, 512, 96), (2048, 136, 4096), (1300, 4096, 256)])
def test_linear_f32_and_grad_match_float64(m, n, k):
    from quant_models import ops

    x, w, b, gy = _inputs(m, n, k)
    parts = w.abs().max().reshape(1)
    y, scale = ops.linear_f32(x, w, b, parts)
    gx, gw = ops.linear_f32_grad(gy, x, w, parts, scale)
    xd, wd, gd = x.double(), w.double(), gy.double()
    wmax = float(wd.abs().max())
    rowx, rowg = xd.abs().amax(1, keepdim=True), gd.abs().amax(1, keepdim=True)
    ey = xd @ wd.t() + b.double()
    assert bool(((y.double() - ey).abs() <= _bound(xd, wd.t(), k, k * 2.0 ** -38 * rowx * wmax) + 2.0 ** -23 * ey.abs()).all())
    assert bool(((gx.double() - gd @ wd).abs() <= _bound(gd, wd, n, n * 2.0 ** -38 * rowg * wmax)).all())
    big = float((rowx * rowg).max())
    assert bool(((gw.double() - gd.t() @ xd).abs() <= _bound(gd.t(), xd, m, m * 2.0 ** -38 * big)).all())


@pytest.mark.gpu
def test_linear_f32_rows_of_any_magnitude():
    """Row scales from 2^-100 to 2^100 and zero rows: every row of y and gx
    keeps its own accuracy; gw that of the largest rows."""
    from quant_models import ops

    m, n, k = 200, 72, 104
    x, w, _, gy = _inputs(m, n, k)
    e = torch.linspace(-100, 60, m, device=DEV).round().reshape(-1, 1)
    x, gy = x * torch.exp2(e), gy * torch.exp2(-e)
    x[::7], gy[::5] = 0, 0
    parts = w.abs().max().reshape(1)
    y, scale = ops.linear_f32(x, w, None, parts)
    gx, gw = ops.linear_f32_grad(gy, x, w, parts, scale)
    xd, wd, gd = x.double(), w.double(), gy.double()
    wmax = float(wd.abs().max())
    assert bool(((y.double() - xd @ wd.t()).abs() <= _bound(xd, wd.t(), k, k * 2.0 ** -38 * xd.abs().amax(1, keepdim=True) * wmax)).all())
    assert bool(((gx.double() - gd @ wd).abs() <= _bound(gd, wd, n, n * 2.0 ** -38 * gd.abs().amax(1, keepdim=True) * wmax)).all())
    big = float((xd.abs().amax(1) * gd.abs().amax(1)).max())
    assert bool(((gw.double() - gd.t() @ xd).abs() <= _bound(gd.t(), xd, m, m * 2.0 ** -38 * big)).all())
    assert not y[::7].any() and not gx[::5].any()


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["feature", "half", "weight"])
def test_linear_f32_values_far_below_a_scale(what):
    """Values 2^0 .. 2^70 below the largest of their scale, in outputs whose
    weights take the largest out: the bar of a float32 product, without a
    floor.  feature: one column of x and gy; half: the first half of their
    columns; weight: columns of w below another part."""
    from quant_models import ops

    m, n, k = 213, 264, 520
    x, w, b, gy = _inputs(m, n, k)
    e = torch.exp2((torch.arange(m, device=DEV) % 71).float()).reshape(-1, 1)
    parts = w.abs().max().reshape(1)
    if what == "feature":
        x[:, 7:8] *= e
        gy[:, 5:6] *= e
        w[:, 7] = w[5] = 0
    elif what == "half":
        x[:, : k // 2] *= e
        gy[:, : n // 2] *= e
        w[: n // 2, : k // 2] = w[: n // 2, k // 4 :] = 0
        w[n // 2 :, : k // 2] = 0
    else:
        x[:, ::2], gy[:, ::2] = 0, 0
        w[:, 1::2] *= 2.0 ** -33
        w[1::2] *= 2.0 ** -33
        parts = torch.stack((w.abs().max(), w[1::2, 1::2].abs().max()))
    y, scale = ops.linear_f32(x, w, None, parts)
    gx, _ = ops.linear_f32_grad(gy, x, w, parts, scale)
    xd, wd, gd = x.double(), w.double(), gy.double()
    assert bool(((y.double() - xd @ wd.t()).abs() <= _bound(xd, wd.t(), k, 0)).all())
    assert bool(((gx.double() - gd @ wd).abs() <= _bound(gd, wd, n, 0)).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(40, 8, 16), (1037, 136, 264), (9000, 72, 104)])
def test_weight_gradient_of_rows_of_any_magnitude(m, n, k):
    """x and grad_y rows of independent magnitudes, products of maxima over
    2^0 .. 2^-80, and columns of x that only the lesser half of the rows have:
    the bar of a float32 product in every column, the same bits each time."""
    from quant_models import ops

    x, w, _, gy = _inputs(m, n, k)
    g = torch.Generator(device=DEV).manual_seed(m)
    ex, eg = (torch.randint(-40, 1, (m, 1), device=DEV, generator=g).float() for _ in range(2))
    x, gy = x * torch.exp2(ex), gy * torch.exp2(eg)
    x[(ex + eg > -40).reshape(-1), : k // 4] = 0
    parts = w.abs().max().reshape(1)
    _, scale = ops.linear_f32(x, w, None, parts)
    _, gw = ops.linear_f32_grad(gy, x, w, parts, scale, want_x=False)
    xd, gd = x.double(), gy.double()
    assert bool(((gw.double() - gd.t() @ xd).abs() <= _bound(gd.t(), xd, m, 0)).all())
    for _ in range(3):
        assert torch.equal(gw, ops.linear_f32_grad(gy, x, w, parts, scale, want_x=False)[1])


@pytest.mark.gpu
def test_ordinary_rows_take_the_split_product():
    """Activations, GELU outputs, quantized rows with few levels left, softmax
    gradients and rows with some outliers are not summed apart: the scales of
    such rows stay positive."""
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(0)
    k = 768
    z = torch.randn(2000, k, device=DEV, generator=g)
    outlier = z.clone()
    outlier[:, 11] *= 1000
    quantized = torch.round(z / z.abs().amax(1, keepdim=True) * 7) * (z.abs().amax(1, keepdim=True) / 7)
    quantized[:, ::2] *= z[:, ::2].abs() > 2.5
    p = torch.softmax(2 * z, 1)
    p[:, 5] -= 1
    for x in (z, torch.nn.functional.gelu(2 * z - 2), outlier, quantized, p, z * (z > 1), z[:, :1].expand(-1, k).contiguous()):
        _, scale = ops.linear_f32(x, z[:8].contiguous(), None, z[:8].abs().max().reshape(1))
        assert bool((scale > 0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("where", ["x", "gy", "w"])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 3.0e38])
def test_linear_f32_special_values(where, value):
    """inf, NaN and the largest floats come out as in a float32 product."""
    from quant_models import ops

    x, w, b, gy = _inputs(150, 40, 64)
    t = {"x": x, "gy": gy, "w": w}[where]
    t[5, 3] = value
    parts = w.abs().max().reshape(1)
    y, scale = ops.linear_f32(x, w, b, parts)
    gx, gw = ops.linear_f32_grad(gy, x, w, parts, scale)
    xc, wc, gc = x.cpu(), w.cpu(), gy.cpu()
    for got, ref in ((y, xc @ wc.t() + b.cpu()), (gx, gc @ wc), (gw, gc.t() @ xc)):
        got = got.cpu()
        assert torch.equal(torch.isnan(got), torch.isnan(ref))
        assert torch.equal(torch.isinf(got), torch.isinf(ref))
        assert torch.equal(got[torch.isinf(got)], ref[torch.isinf(ref)])


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(1, 8, 8), (127, 120, 24), (129, 136, 40), (700, 264, 776), (1300, 1000, 128),
                                   (3000, 16, 4096)])
def test_exact_rows_match_float64(m, n, k):
    """The plain float32 products, at the edges of their 128 x 128 tiles: every
    row where w has no finite bound, single rows with an inf, and all of gw
    beside one.  Each of the con additions of an output rounds once."""
    from quant_models import ops

    x, w, b, gy = _inputs(m, n, k)
    xd, wd, gd = x.double(), w.double(), gy.double()
    none = torch.full((1,), float("inf"), device=DEV)
    y, scale = ops.linear_f32(x, w, b, none)
    gx, _ = ops.linear_f32_grad(gy, x, w, none, scale)
    for got, ref, con, mag in ((y, xd @ wd.t() + b.double(), k, xd.abs() @ wd.abs().t() + b.abs()),
                               (gx, gd @ wd, n, gd.abs() @ wd.abs())):
        assert bool(((got.double() - ref).abs() <= (con + 2) * 2.0 ** -24 * mag).all())
    some = torch.unique(torch.linspace(0, m - 1, 5).long())
    x[some, 3] = float("inf")
    y, scale = ops.linear_f32(x, w, b, w.abs().max().reshape(1))
    _, gw = ops.linear_f32_grad(gy, x, w, w.abs().max().reshape(1), scale)
    assert torch.equal(y[some.cuda()].isinf(), (x[some] @ w.t()).isinf()) and bool(y[some.cuda()].isinf().any())
    keep = [i for i in range(k) if i != 3]
    assert not gw[:, 3].isfinite().any()
    ref = gd.t() @ xd
    assert bool(((gw.double() - ref).abs() <= (m + 2) * 2.0 ** -24 * (gd.abs().t() @ xd.abs()))[:, keep].all())


@pytest.mark.gpu
def test_a_step_of_nan_costs_a_few_ordinary_steps():
    """NaN in every row: all three products in plain float32, 16 times the
    matrix work, which must not become a serial sum per output."""
    from quant_models import ops

    x, w, b, gy = _inputs(12608, 3072, 768)
    parts = w.abs().max().reshape(1)

    def step():
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        y, scale = ops.linear_f32(x, w, b, parts)
        grads = ops.linear_f32_grad(gy, x, w, parts, scale)
        end.record()
        torch.cuda.synchronize()
        return start.elapsed_time(end), (y, *grads)

    usual = min(step()[0] for _ in range(5))
    x[:, 0] = gy[:, 0] = float("nan")
    times, outs = zip(*(step() for _ in range(2)))
    assert all(bool(t.isnan().any()) for t in outs[0])
    assert min(times) <= 16 * usual


@pytest.mark.gpu
def test_linear_f32_empty_gradient():
    from quant_models import ops

    x, w, _, gy = _inputs(130, 24, 48)
    parts = w.abs().max().reshape(1)
    _, scale = ops.linear_f32(x, w, None, parts)
    gx, gw = ops.linear_f32_grad(torch.zeros_like(gy), x, w, parts, scale)
    assert not gx.any() and not gw.any()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(1, 8), (5, 40), (96, 520), (1025, 1000), (4099, 2056), (12608, 3072), (130, 4096)])
def test_bias_gradient_is_the_column_sum(m, n):
    """Each column within the roundings of its additions: a lane's rows, the
    block's 4 waves, 16 partial rows and 6 levels of a tree, 2^-24 each."""
    from quant_models import ops

    x, w, _, gy = _inputs(m, n, 64)
    gy = gy * torch.exp2(torch.randint(-20, 20, (1, n), device=DEV).float())
    parts = w.abs().max().reshape(1)
    _, scale = ops.linear_f32(x, w, None, parts)
    gb = torch.empty(n, device=DEV)
    gx, gw = ops.linear_f32_grad(gy, x, w, parts, scale, grad_b=gb)
    gx0, gw0 = ops.linear_f32_grad(gy, x, w, parts, scale)
    assert torch.equal(gx, gx0) and torch.equal(gw, gw0)
    adds = m // 4096 + 2 + 4 + 16 + 6
    assert bool(((gb.double() - gy.double().sum(0)).abs() <= adds * 2.0 ** -24 * gy.double().abs().sum(0)).all())
    gy[m // 2, 3], gy[0, 5], gy[m - 1, 7] = float("inf"), float("nan"), float("-inf")
    ops.linear_f32_grad(gy, x, w, parts, scale, grad_b=gb)
    assert gb[3] == float("inf") and torch.isnan(gb[5]) and gb[7] == float("-inf")


def _layer(method, act, rot, seed=3):
    from quant_models.quant_i import QATLinearComplexPhase

    torch.manual_seed(seed)
    return QATLinearComplexPhase(method, method, act > 0, max(2, act), rot, in_features=1024, out_features=1536).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("method,act,rot", [("complex_phase_v2", 4, False), ("complex_phase_v1", 0, True),
                                            ("complex_phase_new_v2", 8, True), ("complex_phase_v4", 0, False)])
def test_training_layer_takes_the_split_product(method, act, rot, monkeypatch):
    """The layer's float32 training step on the split kernels against the
    same step on torch's product: float32 rounding, 2^-17 of the largest."""
    from quant_models import quant_i

    layer = _layer(method, act, rot)
    x0 = torch.randn(4, 400, 1024, device=DEV)
    gy = torch.randn(4, 400, 1536, device=DEV)
    calls, real = [], quant_i._SplitLinearFn.apply
    monkeypatch.setattr(quant_i._SplitLinearFn, "apply", lambda *a: calls.append(1) or real(*a))
    out = []
    for limit in (0, float("inf")):
        monkeypatch.setattr(quant_i, "SPLIT_LINEAR_MIN", limit)
        x = x0.clone().requires_grad_(True)
        layer.zero_grad(set_to_none=True)
        y = layer(x)
        y.backward(gy)
        out.append([y.detach(), x.grad] + [p.grad for p in layer.parameters()])
    assert len(calls) == 1
    for a, b in zip(*out):
        assert a.shape == b.shape
        # a rotation's gradient sums 1.5 M products of cancelling signs
        assert float((a - b).abs().max()) <= (2.0 ** -10 if a.numel() == 1 else 2.0 ** -17) * float(b.abs().max())


@pytest.mark.gpu
def test_training_layer_double_backward_and_forward_mode():
    """create_graph gradients of the split product, and forward-mode
    differentiation (which keeps F.linear)."""
    layer = _layer("complex_phase_v2", 0, False)
    x = torch.randn(2000, 1024, device=DEV, requires_grad=True)
    gy = torch.randn(2000, 1536, device=DEV, requires_grad=True)
    (gx,) = torch.autograd.grad(layer(x), x, gy, create_graph=True)
    (ggy,) = torch.autograd.grad(gx, gy, torch.ones_like(gx))
    a = layer.quantized_weight().detach()
    assert torch.allclose(gx.detach(), gy.detach() @ a, rtol=1e-4, atol=1e-4)
    assert torch.allclose(ggy, torch.ones_like(gx) @ a.t(), rtol=1e-4, atol=1e-4)
    for p in layer.parameters():
        p.requires_grad_(False)
    with torch.autograd.forward_ad.dual_level():
        t = torch.randn_like(x)
        y = layer(torch.autograd.forward_ad.make_dual(x.detach(), t))
        ty = torch.autograd.forward_ad.unpack_dual(y).tangent
    assert torch.allclose(ty, t @ a.t(), rtol=1e-4, atol=1e-4)


def test_transformed_gradients_take_torch_products(monkeypatch):
    """Batched gradients (is_grads_batched, vmap) and dual ones reach the
    backward as tensors without memory of their own: torch's products, as
    behind F.linear."""
    from quant_models import ops
    from quant_models.quant_i import _SplitLinearFn

    monkeypatch.setattr(ops, "linear_f32", lambda x, w, b, parts: (torch.nn.functional.linear(x, w, b), x.new_ones(len(x))))
    monkeypatch.setattr(ops, "linear_f32_grad", lambda *a: pytest.fail("the kernels were given a transformed gradient"))
    x, w, b, _ = (t.requires_grad_(True) for t in _inputs(6, 4, 8, dev="cpu"))
    gys = torch.randn(3, 6, 4)
    y = _SplitLinearFn.apply(x, w, b, torch.ones(1))
    ref = torch.nn.functional.linear(x, w, b)
    want = torch.autograd.grad(ref, (x, w, b), gys, is_grads_batched=True, retain_graph=True)
    got = torch.autograd.grad(y, (x, w, b), gys, is_grads_batched=True, retain_graph=True)
    mapped = torch.func.vmap(lambda g: torch.autograd.grad(y, (x, w, b), g, retain_graph=True))(gys)
    for a, c, d in zip(want, got, mapped):
        assert torch.allclose(a, c) and torch.allclose(a, d)
    with torch.autograd.forward_ad.dual_level():
        g = torch.autograd.forward_ad.make_dual(gys[0], gys[1])
        for a, c in zip(torch.autograd.grad(y, (x, w, b), g), torch.autograd.grad(ref, (x, w, b), g)):
            a, c = torch.autograd.forward_ad.unpack_dual(a), torch.autograd.forward_ad.unpack_dual(c)
            assert torch.allclose(a.primal, c.primal) and torch.allclose(a.tangent, c.tangent)


@pytest.mark.gpu
def test_split_product_in_a_captured_graph():
    """Forward and gradients captured once and replayed on other operands, some
    with rows that are summed apart: every replay gives the eager bits."""
    from quant_models import ops

    x, w, b, gy = _inputs(1500, 136, 264)
    parts, gb = w.abs().max().reshape(1), torch.empty(136, device=DEV)

    def step():
        y, scale = ops.linear_f32(x, w, b, parts)
        return (y, *ops.linear_f32_grad(gy, x, w, parts, scale, grad_b=gb), gb)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = step()
    for k in range(5):
        x.normal_()
        gy.normal_()
        if k == 1:
            x[5, 3], gy[7, 9] = float("nan"), float("inf")
        if k == 2:
            x[11, 7], gy[900:] = 2.0 ** 25, gy[900:] * 2.0 ** -30
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in outs]
        for a, c in zip(got, step()):
            assert torch.equal(a.view(torch.int32), c.view(torch.int32)) or torch.equal(a.nan_to_num(7.0), c.nan_to_num(7.0))


@pytest.mark.gpu
def test_operands_that_do_not_fit_are_refused():
    """By F.linear's own error from the layer, by the host checks below it."""
    from quant_models import ops

    layer = _layer("complex_phase_v2", 0, False)
    for shape in ((4096, 1016), (4096, 2048)):
        with pytest.raises(RuntimeError):
            layer(torch.randn(*shape, device=DEV))
    layer.bias = torch.nn.Parameter(torch.zeros(1528, device=DEV))
    with pytest.raises(RuntimeError):
        layer(torch.randn(4096, 1024, device=DEV))
    x, w, b, gy = _inputs(64, 40, 48)
    parts = w.abs().max().reshape(1)
    y, scale = ops.linear_f32(x, w, b, parts)
    for args in ((x[:, :40], w, b), (x, w, b[:32]), (x.half(), w, b), (x, w.t().contiguous().t(), b)):
        with pytest.raises(ValueError):
            ops.linear_f32(*args, parts)
    for args in ((gy[:32], x), (gy, x[:, :40]), (gy, x.half()), (gy.t().contiguous().t(), x)):
        with pytest.raises(ValueError):
            ops.linear_f32_grad(*args, w, parts, scale)


def _pays(m, n, k, grad=True):
    from types import SimpleNamespace

    from quant_models import quant_i

    x = SimpleNamespace(dim=lambda: 2, shape=(m, k), numel=lambda: m * k, device=SimpleNamespace(type="cuda"), is_cuda=True,
                        dtype=torch.float32, requires_grad=False)
    w = SimpleNamespace(shape=(n, k), device=x.device, dtype=torch.float32, is_contiguous=lambda: True, data_ptr=lambda: 256,
                        requires_grad=grad)
    return quant_i._split_linear_pays(x, w, None)


def test_split_product_leaves_narrow_layers_to_the_library():
    """Layers whose splits move more than the products save."""
    assert _pays(401408, 288, 96) and _pays(100352, 192, 192) and _pays(100352, 192, 768, grad=False)
    for m, n, k in ((1 << 20, 64, 64), (1 << 19, 384, 32), (1 << 19, 32, 384), (150000, 1024, 16), (1 << 17, 8, 4096)):
        assert 2 * m * n * k > 4.5e9 and not _pays(m, n, k)
    assert not _pays(401408, 96, 384, grad=False)
    with torch.no_grad():
        assert not _pays(401408, 96, 384) and _pays(12608, 3072, 768)


def test_split_product_scratch():
    """The workspace is the operands' planes and little else, and a layer whose
    planes pass the limit keeps F.linear, which needs none."""
    from quant_models import _native as N

    lib, m, n, k = N.load(), 496, 4096, 4096  # one split of grad_w
    planes = 4 * 768 * (n + k) + 4 * n * k  # x, grad_y (768 padded rows), w
    assert planes <= lib.rpfq_linear_f32_workspace_bytes(m, n, k, 1) <= planes + (1 << 20)
    assert lib.rpfq_linear_f32_workspace_bytes(m, n, k, 0) <= planes
    # the column sums of the bias gradient fit where x's planes go
    assert lib.rpfq_linear_f32_workspace_bytes(4096, 4096, 8, 1) >= 1024 * 4096 * 4 + 4096 * 4096 * 4

    assert _pays(12608, 3072, 768) and _pays(1 << 18, 3072, 768)
    assert not _pays(12608, 4104, 768) and not _pays(12608, 768, 4104)  # past the kernels' columns
    assert not _pays(1 << 19, 3072, 768) and not _pays(1 << 24, 4096, 4096) and not _pays(4096, 3072, 0)


def test_split_product_switch():
    """RPFQ_SPLIT_LINEAR=0 leaves every training product to F.linear."""
    import os
    import subprocess
    import sys

    from quant_models import _native as N

    for value, limit in (("0", "inf"), ("1", "4500000000.0")):
        env = dict(os.environ, RPFQ_SPLIT_LINEAR=value, PYTHONPATH=os.path.dirname(os.path.dirname(N.__file__)))
        out = subprocess.run([sys.executable, "-c", "from quant_models import quant_i; print(quant_i.SPLIT_LINEAR_MIN)"],
                             env=env, capture_output=True, text=True, timeout=300)
        assert out.stdout.strip() == limit, out.stderr


def test_linear_f32_argument_errors():
    """Reported on the host, without a GPU."""
    from quant_models import _native as N

    lib = N.load()
    p = ctypes.c_void_p(4096)
    assert lib.rpfq_linear_f32_workspace_bytes(64, 64, 64, 0) > 64 * 64 * 4
    for m, n, k in ((0, 64, 64), (64, 60, 64), (64, 64, 4104), (1 << 25, 64, 64)):
        assert lib.rpfq_linear_f32_workspace_bytes(m, n, k, 1) == 0
        assert lib.rpfq_linear_f32(p, p, None, m, n, k, p, 1, p, p, p, 1 << 30, None) == 2
    assert lib.rpfq_linear_f32(p, None, None, 64, 64, 64, p, 1, p, p, p, 1 << 30, None) == 1
    assert lib.rpfq_linear_f32(p, p, None, 64, 64, 64, p, 0, p, p, p, 1 << 30, None) == 6
    assert lib.rpfq_linear_f32(p, p, None, 64, 64, 64, p, 1, p, p, p, 1024, None) == 2
    assert lib.rpfq_linear_f32(ctypes.c_void_p(4100), p, None, 64, 64, 64, p, 1, p, p, p, 1 << 30, None) == 3
    assert lib.rpfq_linear_f32_grad(p, p, p, 64, 64, 64, p, 1, p, None, None, p, p, 1 << 30, None) == 1


def test_row_and_weight_scales_hold_the_bound():
    """The float32 A_q of every method stays below the sum of its scales
    (what scales w in rpfq_linear_f32), also rotated."""
    from oracle import rpfq_oracle as O

    rng = np.random.default_rng(0)
    w = rng.standard_normal((64, 48)).astype(np.float32)
    for kind, steps in (("axis", 1), ("axis", 2), ("axis", 4), ("sign", 2)):
        for t in (0.0, 0.7, -1.9):
            cs = (np.float32(np.cos(t)), np.float32(np.sin(t)))
            a, su, sw = O.quantized_weight(w, kind, steps, kind, steps, (cs, cs) if t else None)
            total = sum(float(abs(s_re)) + float(abs(s_im)) for _, s_re, s_im in su + sw)
            assert np.abs(a).max() <= total * (1 + 2.0 ** -20)
