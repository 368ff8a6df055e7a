"""rpfq_attention against float64 softmax(q k^T scale) v.

Bar: every probability and the output are rounded once to 16 bits (2^-11 or
2^-8 relative) and the probabilities sum to 1, so an output is within
2.5 u max|v| of the exact one; the float32 scores add at most
2^-20 |q| |k| scale in the exponent.
"""
import ctypes

import pytest
import torch

DEV = "cuda"


def _exact(qkv, heads, scale):
    b, n, c3 = qkv.shape
    q, k, v = (t.contiguous() for t in qkv.double().reshape(b, n, 3, heads, 64).permute(2, 0, 3, 1, 4).unbind(0))
    p = torch.softmax(q @ k.transpose(-1, -2).contiguous() * scale, -1)
    return (p @ v).transpose(1, 2).reshape(b, n, c3 // 3)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,n,heads", [(1, 1, 1), (2, 31, 2), (1, 32, 3), (3, 33, 1), (2, 64, 2), (2, 65, 1), (2, 128, 1),
                                       (1, 129, 2), (1, 160, 1), (1, 161, 3), (2, 192, 1), (40, 197, 12), (1, 225, 2),
                                       (1, 257, 16), (2, 288, 1)])
def test_attention_matches_float64(b, n, heads, dtype):
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(n)
    qkv = (torch.randn(b, n, 3 * heads * 64, device=DEV, generator=g) * 1.5).to(dtype)
    out = ops.attention(qkv, heads, 0.125)
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    err = (out.double() - _exact(qkv, heads, 0.125)).abs().max()
    assert out.shape == (b, n, heads * 64) and out.dtype == dtype
    assert float(err) <= (2.5 * u + 2.0 ** -13) * float(qkv.abs().max())


@pytest.mark.gpu
def test_attention_extreme_scores_and_special_values():
    """Scores far apart (one probability near 1), an unaligned view, and inf /
    NaN in v reach the outputs of their head and image only."""
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(1)
    n, heads = 197, 2
    qkv = torch.randn(2, n, 3 * heads * 64, device=DEV, generator=g).half()
    qkv[..., : 2 * heads * 64] *= 12
    ref = _exact(qkv, heads, 0.125)
    assert float((ops.attention(qkv, heads, 0.125).double() - ref).abs().max()) <= 2.5 * 2.0 ** -11 * float(qkv[..., 2 * heads * 64:].abs().max())
    flat = torch.zeros(qkv.numel() + 1, device=DEV, dtype=torch.float16)
    flat[1:] = qkv.reshape(-1)
    assert torch.equal(ops.attention(flat[1:].view_as(qkv), heads, 0.125), ops.attention(qkv, heads, 0.125))
    base = torch.randn(2, n, 3 * heads * 64, device=DEV, generator=g).half()
    for value in (float("inf"), float("-inf"), float("nan")):
        qkv = base.clone()
        qkv[1, n - 1, 2 * heads * 64 + 5] = value  # v of the last token, image 1, head 0, value 5
        out, clean = ops.attention(qkv, heads, 0.125), ops.attention(base, heads, 0.125)
        hit = torch.zeros_like(out, dtype=torch.bool)
        hit[1, :, 5] = True
        assert torch.equal(out[~hit], clean[~hit])
        got = out[hit]
        assert bool(torch.isnan(got).all()) if value != value else bool((got == value).all())


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 20, 31, 32, 33, 63, 64, 65, 82, 95, 96, 97, 127, 129, 161, 193, 225, 288])
def test_attention_special_values_at_every_padding(n):
    """inf and NaN in v of the first and last token, 0 to 63 rows of padding
    behind it: that output column only, and never NaN from an inf."""
    from quant_models import ops

    heads = 2
    base = torch.randn(2, n, 3 * heads * 64, device=DEV, generator=torch.Generator(device=DEV).manual_seed(n)).half()
    clean = ops.attention(base, heads, 0.125)
    for token in (0, n - 1):
        for value in (float("inf"), float("-inf"), float("nan")):
            qkv = base.clone()
            qkv[1, token, 2 * heads * 64 + 64 + 37] = value  # image 1, head 1, value 37
            out = ops.attention(qkv, heads, 0.125)
            got = out[1, :, 64 + 37].clone()
            assert bool(torch.isnan(got).all()) if value != value else bool((got == value).all())
            out[1, :, 64 + 37] = clean[1, :, 64 + 37]
            assert torch.equal(out, clean)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,size", [(torch.float16, 32.0), (torch.bfloat16, 32.0), (torch.bfloat16, 2.0 ** 40)])
@pytest.mark.parametrize("n", [5, 64, 197, 288])
def test_attention_scores_past_the_float32_integers(n, dtype, size):
    """Finite scores of any size: q and k are small integers times `size`, so
    float32 holds each score exactly, and every row that has its own key wins
    by far.  The largest scores, times scale and log2(e), pass 2^24 (bf16:
    2^85), where float32 has no fractions left."""
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(n)
    heads = 2
    qkv = torch.randint(-63, 64, (2, n, 3, heads, 64), device=DEV, generator=g).float() * size
    far = torch.arange(1, n + 1, device=DEV).reshape(1, n, 1, 1) % 31 + 32.0
    sign = torch.randint(0, 2, (2, n, heads, 64), device=DEV, generator=g) * 2.0 - 1
    qkv[:, :, 0] = qkv[:, :, 1] = sign * far * size
    qkv[:, :, 2] = torch.randn(2, n, heads, 64, device=DEV, generator=g)
    qkv = qkv.reshape(2, n, -1).to(dtype)
    ref = _exact(qkv, heads, 0.125)
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    out = ops.attention(qkv, heads, 0.125).double()
    assert bool(out.isfinite().all())
    assert float((out - ref).abs().max()) <= 2.5 * u * float(qkv.reshape(2, n, 3, -1)[:, :, 2].abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 64, 197, 288])
def test_attention_of_the_largest_bf16_values(n):
    """v up to bf16's largest: a weighted mean of finite values is finite."""
    from quant_models import ops

    g = torch.Generator(device=DEV).manual_seed(n)
    qkv = torch.randn(2, n, 3 * 64, device=DEV, generator=g)
    qkv[..., 128:] = 1.5 * 2.0 ** 126 + 2.0 ** 125 * torch.rand(2, n, 64, device=DEV, generator=g)
    qkv[..., 150:] *= -1
    qkv = qkv.bfloat16()
    out = ops.attention(qkv, 1, 0.125).double()
    assert bool(out.isfinite().all())
    assert float((out - _exact(qkv, 1, 0.125)).abs().max()) <= 2.5 * 2.0 ** -8 * float(qkv.abs().max())


@pytest.mark.gpu
def test_block_attention_route():
    """The block's attention takes the kernel in inference only, and agrees
    with torch's there."""
    from quant_models import ops
    from quant_models.inference import load_synthetic_codes, prepare_inference
    from quant_models.quant_rpfq_vit import ComplexVisionTransformer

    torch.manual_seed(0)
    model = ComplexVisionTransformer(img_size=32, embed_dim=192, depth=1, num_heads=3, enable_act_quant=False,
                                     enable_rotation=False)
    load_synthetic_codes(model, 1)
    attn = prepare_inference(model).blocks[0].attn
    calls, real = [], ops.attention
    ops.attention = lambda *a: calls.append(1) or real(*a)
    try:
        x = torch.randn(2, 50, 192, device=DEV).half()
        with torch.no_grad():
            y = attn(x)
            qkv = attn.qkv(x)
            q, k, v = qkv.reshape(2, 50, 3, 3, 64).permute(2, 0, 3, 1, 4).unbind(0)
            ref = torch.nn.functional.scaled_dot_product_attention(q, k, v).transpose(1, 2).reshape(2, 50, 192)
            assert torch.allclose(attn._attend(qkv), ref, rtol=2.0 ** -9, atol=2.0 ** -9 * float(v.abs().max()))
            assert len(calls) == 2 and y.shape == x.shape
            attn(torch.randn(1, 289, 192, device=DEV).half())  # too many tokens
            with torch.autocast("cuda", dtype=torch.bfloat16):  # torch's runs in the autocast dtype
                assert attn._attend(qkv).dtype == torch.bfloat16
            assert len(calls) == 2
        for p in attn.parameters():
            p.requires_grad_(False)
        xg = x.clone().requires_grad_(True)
        attn(xg).sum().backward()
        assert xg.grad is not None and len(calls) == 2
    finally:
        ops.attention = real


def test_block_attention_keeps_torch_outside_the_kernels_limits():
    """Every size and scale that torch's attention takes is still taken: the
    kernel's limits choose the route, and both routes use the same scale."""
    from types import SimpleNamespace

    from quant_models.vision_transformer import Attention

    def takes(b, n, heads, scale=None):
        attn = Attention(64 * heads, heads).eval()
        attn.qkv.use_packed = True
        attn.scale = attn.scale if scale is None else scale
        qkv = SimpleNamespace(is_cuda=True, dtype=torch.float16, requires_grad=False, shape=(b, n, 192 * heads))
        return attn._attends_on_device(qkv)

    assert takes(256, 197, 12) and takes(1 << 24, 1, 1) and takes(4, 288, 3, 2.5)
    assert not takes((1 << 24) + 1, 1, 1) and not takes(1 << 23, 2, 3) and not takes(1, 289, 1)
    for scale in (0.0, -0.125, float("inf"), float("nan")):
        assert not takes(1, 8, 1, scale)
    attn = Attention(128, 2).eval()
    qkv = torch.randn(2, 9, 384, generator=torch.Generator().manual_seed(0))
    q, k, v = qkv.reshape(2, 9, 3, 2, 64).permute(2, 0, 3, 1, 4).unbind(0)
    for attn.scale in (0.125, 0.5, 0.0, -0.25):
        ref = (torch.softmax(q @ k.transpose(-1, -2) * attn.scale, -1) @ v).transpose(1, 2).reshape(2, 9, 128)
        assert torch.allclose(attn._attend(qkv), ref, rtol=1e-5, atol=1e-5)


def test_attention_argument_errors():
    from quant_models import _native as N

    lib = N.load()
    p = ctypes.c_void_p(4096)
    assert lib.rpfq_attention(None, N.F16, 1, 8, 1, 64, 0.125, p, None) == 1
    assert lib.rpfq_attention(p, N.F32, 1, 8, 1, 64, 0.125, p, None) == 5
    for b, n, h, d in ((0, 8, 1, 64), (1, 289, 1, 64), (1, 8, 1, 32), (1, 8, 2048, 64)):
        assert lib.rpfq_attention(p, N.F16, b, n, h, d, 0.125, p, None) == 2
    assert lib.rpfq_attention(ctypes.c_void_p(4098), N.F16, 1, 8, 1, 64, 0.125, p, None) == 3
    for scale in (0.0, -0.125, float("nan"), float("inf")):
        assert lib.rpfq_attention(p, N.F16, 1, 8, 1, 64, scale, p, None) == 6


def test_attention_refuses_heads_that_do_not_divide_the_row():
    """387 values are not 3 x 2 heads of 64: the kernel would walk shorter
    tokens than there are."""
    from quant_models import ops

    for shape, heads in (((2, 20, 387), 2), ((2, 20, 384), 0), ((2, 20, 384), 5), ((20, 384), 2)):
        with pytest.raises(ValueError, match="heads"):
            ops.attention(torch.zeros(*shape, dtype=torch.half), heads, 0.125)
