"""Activation quantization into prescaled fp16 rows in one pass
(rpfq_act_quant_prescaled) against its two passes, bit for bit."""
import ctypes

import pytest
import torch

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bits", [2, 4, 8, 16])
@pytest.mark.parametrize("m,c", [(1, 16), (257, 96), (130, 272), (1500, 528), (2051, 768), (300, 2064), (131, 3088), (64, 4096)])
def test_equals_act_quant_then_prescale(m, c, bits, dtype):
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(m + c + bits)
    x = torch.randn(m, c, device=DEV, generator=g)
    x *= torch.exp2(torch.randint(-40, 41, (m, 1), device=DEV, generator=g).float())
    x[::5] = 0
    x[m // 2, c // 2:] = 0
    if m > 4:
        x[1, 3], x[2, 5], x[3, c - 1] = float("inf"), float("nan"), 3e38
    x = x.to(dtype)
    y, s = ops.act_quant_prescaled(x, bits)
    y2, s2 = ops.prescale_rows(ops.act_quant(x, bits))
    assert torch.equal(s.view(torch.int32), s2.view(torch.int32))
    nan = torch.isnan(y2)
    assert torch.equal(torch.isnan(y), nan)
    assert torch.equal(y.view(torch.int16)[~nan], y2.view(torch.int16)[~nan])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("form", ["rows", "strided", "offset"])
def test_layer_forms_keep_their_bits(dtype, form, monkeypatch):
    """forward, forward_gelu and forward_residual of a layer whose launch the
    DMA kernel takes: the one pass is used and the results stay."""
    from quant_models import ops
    from quant_models.quant_i import QATLinearComplexPhase

    torch.manual_seed(1)
    layer = QATLinearComplexPhase("complex_phase_v2", "complex_phase_v2", True, 4, True, in_features=384,
                                  out_features=768).to(DEV).eval()
    layer.use_packed = True
    x = torch.randn(9000, 384, device=DEV).to(dtype)
    if form == "strided":
        x = x.t().contiguous().t()
    elif form == "offset":
        x = torch.zeros(9000 * 384 + 1, device=DEV, dtype=dtype)[1:].view(9000, 384).copy_(x)
    r = torch.randn(9000, 768, device=DEV).to(dtype)
    calls, real = [], ops.act_quant_prescaled

    def run():
        with torch.no_grad():
            return layer(x), layer.forward_gelu(x), layer.forward_residual(x, r)

    monkeypatch.setattr(ops, "act_quant_prescaled", lambda *a: calls.append(1) or real(*a))
    one = run()
    assert len(calls) == 3
    monkeypatch.setattr(ops.PackedWide, "act_quant_operand", lambda self, x, bits, *a: (ops.act_quant(x, bits), None))
    for a, b in zip(one, run()):
        assert a.dtype == dtype and torch.equal(a, b)


def test_argument_errors():
    from quant_models import _native as N

    f, p = N.load().rpfq_act_quant_prescaled, ctypes.c_void_p(4096)
    assert f(None, N.F32, 4, 64, 4, p, p, None) == 1
    assert f(p, N.F32, 4, 64, 4, p, None, None) == 1
    assert f(p, N.F16, 4, 64, 4, p, p, None) == 5
    for c in (24, 4112):
        assert f(p, N.F32, 4, c, 4, p, p, None) == 2
    assert f(p, N.F32, 4, 64, 4, ctypes.c_void_p(4104), p, None) == 3
    for bits in (1, 17):
        assert f(p, N.F32, 4, 64, bits, p, p, None) == N.load().rpfq_act_quant(p, N.F32, 4, 64, bits, p, N.F32, None)
