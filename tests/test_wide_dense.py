"""The decoded-fragment kernels: rpfq_wide_linear_dense against the packed DMA
kernel (the same bits) and rpfq_wide_linear_grad_x_dense against float64.

Bar of the gradient: grad_y rows carry one fp16 rounding (2^-11 of each
element, or 2^-24 of the row's largest) and the products are summed in
float32, 2^-23 of sum |gy| |A| per 16 terms; the store rounds once more.
"""
import ctypes
import itertools

import pytest
import torch

DEV = "cuda"
ROT = ((0.8, 0.6), (0.6, -0.8))
DTYPES = [torch.float16, torch.bfloat16, torch.float32]


def _layer(n, k, cb, block, rot, seed=0):
    from quant_models import _native as N
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(seed)
    bits, count = (2, 4) if cb in (N.CB_AXIS, N.CB_SIGN) else (4, 2)
    planes = [torch.randint(0, 256, (n, k * bits // 8), generator=g, device=DEV, dtype=torch.uint8) for _ in range(count)]
    cols = 16 if cb == N.CB_TABLE else 1 if block == 0 else -(-k // block)
    sre, sim = ([0.003 + 0.027 * torch.rand(n, cols, generator=g, device=DEV) for _ in range(count)] for _ in range(2))
    return ops.PackedWide.from_planes(planes, sre, sre if cb == N.CB_PSK16 else sim, n, k, cb, 2 if count == 4 else 1,
                                      block, rot), g


def _dense(pw, x, xs, bias, res, out_dtype, gelu):
    from quant_models import _native as N

    lib = N.load()
    nbytes = lib.rpfq_wide_dense_bytes(ctypes.byref(pw.desc), 0)
    assert nbytes > 0
    work = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    y = torch.full((x.shape[0], pw.out_features), 7.0, device=DEV, dtype=out_dtype)
    N.check("dense", lib.rpfq_wide_linear_dense(
        ctypes.byref(pw.desc), pw.blob.data_ptr(), pw.blob.numel(), x.data_ptr(), x.shape[0], N.ptr(xs), N.ptr(bias),
        N.ptr(res), y.data_ptr(), N.dtype_code(out_dtype), N.FLAG_GELU if gelu else 0, work.data_ptr(), nbytes,
        N.stream_of(x)))
    return y


SHAPES = [(128, 16, 32, 0, 0, None), (129, 50, 64, 0, 0, None), (200, 96, 96, 1, 0, ROT), (333, 130, 160, 2, 0, None),
          (1000, 144, 32, 3, 0, None), (777, 258, 128, 0, 32, None), (520, 64, 256, 0, 64, ROT),
          (2500, 500, 384, 0, 0, None), (12608, 384, 64, 0, 0, None)]


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,cb,block,rot", SHAPES)
def test_dense_linear_equals_dma_kernel(m, n, k, cb, block, rot, monkeypatch):
    from quant_models import _native as N
    from quant_models import ops

    monkeypatch.setattr(ops, "DENSE", False)
    pw, g = _layer(n, k, cb, block, rot)
    bias = torch.randn(2 * n, device=DEV, generator=g)
    for dt, out, gelu, res in itertools.product(DTYPES, DTYPES, (False, True), (False, True)):
        if gelu and res:
            continue
        x = torch.randn(m, 2 * k, device=DEV, generator=g).to(dt)
        r = torch.randn(m, 2 * n, device=DEV, generator=g).to(out) if res else None
        b = bias if gelu or res else None
        assert pw.kernel_for(m, torch.float16, out, N.FLAG_NO_STREAM | (N.FLAG_GELU if gelu else 0)) == N.KERNEL_DMA
        x2, xs = (x, None) if dt == torch.float16 else ops.prescale_rows(x)
        want = pw.linear(x2, b, out_dtype=out, flags=N.FLAG_NO_STREAM, residual=r, gelu=gelu, row_scale=xs)
        assert torch.equal(_dense(pw, x2, xs, b, r, out, gelu), want)
        if res:  # in place
            y = r.clone()
            work = torch.empty(N.load().rpfq_wide_dense_bytes(ctypes.byref(pw.desc), 0), dtype=torch.uint8, device=DEV)
            N.check("dense", N.load().rpfq_wide_linear_dense(
                ctypes.byref(pw.desc), pw.blob.data_ptr(), pw.blob.numel(), x2.data_ptr(), m, N.ptr(xs), N.ptr(b),
                y.data_ptr(), y.data_ptr(), N.dtype_code(out), 0, work.data_ptr(), work.numel(), N.stream_of(x2)))
            assert torch.equal(y, want)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,gelu,out", [(3200, 1536, 768, True, torch.float16), (2000, 384, 1536, False, torch.bfloat16),
                                            (1500, 500, 384, False, torch.float16), (1400, 384, 384, False, torch.float32)])
def test_linear_route_gives_the_same_bits(m, n, k, gelu, out, monkeypatch):
    """PackedWide.linear takes the decoded weight for these and returns what
    the DMA kernel returns."""
    from quant_models import ops

    pw, g = _layer(n, k, 0, 0, None)
    x = torch.randn(m, 2 * k, device=DEV, generator=g).to(out)
    r = None if gelu else torch.randn(m, 2 * n, device=DEV, generator=g).to(out)
    y = pw.linear(x, None, residual=r, gelu=gelu)
    assert pw._dense_bytes(m, x.half(), out, 8 if gelu else 0, r is not None) > 0
    monkeypatch.setattr(ops, "DENSE", False)
    assert torch.equal(y, pw.linear(x, None, residual=r, gelu=gelu))


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,cb,block,rot", [(128, 256, 16, 0, 0, None), (129, 1024, 48, 0, 0, None),
                                                (400, 384, 96, 1, 0, ROT), (333, 1024, 136, 2, 0, None),
                                                (2000, 1056, 144, 3, 0, None), (777, 1024, 256, 0, 32, None),
                                                (520, 1024, 64, 0, 64, ROT), (12608, 1536, 384, 0, 0, None)])
def test_dense_grad_x_matches_float64(m, n, k, cb, block, rot):
    from quant_models import _native as N
    from quant_models import ops

    pw, g = _layer(n, k, cb, block, rot)
    a = pw.decode(round_fp16=True).double()
    lib = N.load()
    nbytes = lib.rpfq_wide_dense_bytes(ctypes.byref(pw.desc), 1)
    work = torch.empty(nbytes, dtype=torch.uint8, device=DEV)
    for dt, out in itertools.product(DTYPES, DTYPES):
        low = -6 if dt == torch.float16 else -30
        e = torch.randint(low, 3, (m, 1), device=DEV, generator=g).float()
        gy = (torch.randn(m, 2 * n, device=DEV, generator=g) * torch.exp2(e)).to(dt)
        g2, s = (gy, None) if dt == torch.float16 else ops.prescale_rows(gy)
        gx = torch.empty(m, 2 * k, device=DEV, dtype=out)
        N.check("grad", lib.rpfq_wide_linear_grad_x_dense(
            ctypes.byref(pw.desc), pw.blob.data_ptr(), pw.blob.numel(), g2.data_ptr(), m, N.ptr(s), gx.data_ptr(),
            N.dtype_code(out), work.data_ptr(), nbytes, N.stream_of(g2)))
        gd = gy.double()
        exact, mag = gd @ a, gd.abs() @ a.abs()
        u = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}[out]
        floor = 2.0 ** -24 if out == torch.float16 else 2.0 ** -133
        row = gd.abs().amax(1, keepdim=True) * 2.0 ** -24 * a.abs().sum(0, keepdim=True)
        bound = ((0.0 if dt == torch.float16 else 2.0 ** -11) + (2 * n / 16 + 1) * 2.0 ** -23) * mag + row + u * exact.abs() + floor
        assert bool(((gx.double() - exact).abs() <= bound).all())


@pytest.mark.gpu
@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan")])
def test_dense_grad_x_special_values(value, dt, monkeypatch):
    """inf and NaN in a row of grad_y come out as in a float32 product and, also
    beside values past fp16, as from the adjoint kernel; other rows keep theirs."""
    from quant_models import ops

    pw, g = _layer(1024, 136, 0, 0, None)
    gy = torch.randn(600, 2048, device=DEV, generator=g).to(dt)
    clean = pw.grad_x(gy)
    assert pw._grad_dense_bytes(600, gy) > 0
    gy[3, 70] = value
    gy[599, 1500] = value
    if dt != torch.float16:
        gy[599, 1501] = 1e30  # finite, and past fp16
    gx = pw.grad_x(gy, out_dtype=torch.float32)
    ref = gy.float().cpu() @ pw.decode(round_fp16=True).cpu()
    keep = [i for i in range(600) if i not in (3, 599)]
    assert torch.equal(pw.grad_x(gy)[keep], clean[keep])
    monkeypatch.setattr(ops, "DENSE", False)
    adjoint = pw.grad_x(gy, out_dtype=torch.float32).cpu()
    for r, other in ((3, adjoint), (599, adjoint), (3, ref)):
        got, want = gx[r].cpu(), other[r]
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
        assert torch.equal(got[got.isinf()], want[want.isinf()])


def test_decoded_weight_routes():
    """Where the decoded weight is left to the kernels that decode in their
    loop: few columns over many rows, and gradients of short rows that their
    prescale pass outweighs."""
    from types import SimpleNamespace

    from quant_models import _native as N
    from quant_models import ops

    def routes(m, n, k, dt):
        pw = ops.PackedWide(n, k, N.CB_AXIS, 2, 0, torch.empty(0, dtype=torch.uint8), None)
        half, g = SimpleNamespace(dtype=torch.float16), SimpleNamespace(dtype=dt)
        return pw._dense_bytes(m, half, dt, 0, False) > 0, pw._grad_dense_bytes(m, g) > 0

    for dt in DTYPES:
        assert routes(12608, 384, 1536, dt) == (True, True) and routes(16000, 48, 2048, dt)[0]
        assert not routes(32768, 48, 2048, torch.float16)[0] and not routes(40000, 192, 1024, torch.float16)[0]
        assert routes(50432, 1024, 96, dt)[1] == (dt == torch.float16) and routes(8192, 1536, 96, dt)[1]
    assert not routes(16384, 384, 160, torch.float32)[1] and routes(8192, 768, 128, torch.float32)[1]


def test_dense_argument_errors():
    from quant_models import _native as N
    from quant_models import ops

    lib = N.load()
    p = ctypes.c_void_p(1 << 16)
    d = ops.make_desc(64, 96, N.CB_AXIS, 2, 0, None)
    big = 1 << 30
    assert lib.rpfq_wide_dense_bytes(ctypes.byref(d), 0) == 256 * 192 * 2
    assert lib.rpfq_wide_dense_bytes(ctypes.byref(d), 1) == 256 * 128 * 2
    for n, k in ((64, 40), (33, 96)):
        assert lib.rpfq_wide_dense_bytes(ctypes.byref(ops.make_desc(n, k, N.CB_AXIS, 2, 0, None)), 0) == 0
    args = (ctypes.byref(d), p, big, p, 256)
    assert lib.rpfq_wide_linear_dense(*args, None, None, None, p, N.F16, 2, p, big, None) == 6
    assert lib.rpfq_wide_linear_dense(*args, None, None, p, p, N.F16, N.FLAG_GELU, p, big, None) == 6
    assert lib.rpfq_wide_linear_dense(*args, None, None, None, p, 9, 0, p, big, None) == 5
    assert lib.rpfq_wide_linear_dense(*args, None, None, None, p, N.F16, 0, p, 64, None) == 2
    assert lib.rpfq_wide_linear_dense(*args[:4], 127, None, None, None, p, N.F16, 0, p, big, None) == 2
    assert lib.rpfq_wide_linear_dense(*args, None, None, None, ctypes.c_void_p(8), N.F16, 0, p, big, None) == 3
    assert lib.rpfq_wide_linear_grad_x_dense(*args, None, None, N.F16, p, big, None) == 1
