"""The e4m3 quantiser's kernels give the scale and the codes of the torch
expression bit for bit (fskernels/triton/triton_gqa_decode_hf_fp8.py:13-16)."""
import pytest
import torch

from fskernels.hip import decode as dec

pytestmark = pytest.mark.gpu
DEV = "cuda"


def expression(x):
    scale = x.abs().max().clamp(min=1e-12) / dec.FP8_MAX
    return (x / scale).clamp(-dec.FP8_MAX, dec.FP8_MAX).to(dec.FP8_DTYPE), scale


def check(got, x, what):
    codes, scale = got
    want, ws = expression(x)
    assert codes.dtype == torch.float8_e4m3fn and codes.shape == x.shape and codes.stride() == want.stride(), what
    assert scale.shape == () and scale.dtype == torch.float32, what
    same = torch.equal(scale, ws) or bool(torch.isnan(scale) & torch.isnan(ws))
    assert same, f"{what}: scale {scale.item()} / {ws.item()}"
    assert torch.equal(codes.view(torch.uint8), want.view(torch.uint8)), what


# steps of 16 elements, workgroups of 256 steps, at most 1024 workgroups: one
# element either side of each, and several steps per thread with a tail
@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 4096, 4097, 1024 * 4096 - 16, 1024 * 4096 + 5, 9_000_013])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_codes_match_the_expression(n, dtype):
    g = torch.Generator(device=DEV).manual_seed(n)
    x = torch.randn(n, generator=g, device=DEV).to(dtype)
    check(dec.quantize_each_to_fp8(x)[0], x.float(), f"n={n} {dtype}")
    check(dec.quantize_to_fp8(x.float()), x.float(), f"n={n} fp32 of {dtype}")


def test_values_on_rounding_boundaries():
    """Quotients on and next to every e4m3 rounding boundary, subnormal codes
    and tiny, huge and zero tensors."""
    codes = torch.arange(0, 127, dtype=torch.uint8).view(torch.float8_e4m3fn).float()
    mid = (codes[1:] + codes[:-1]) / 2
    near = torch.cat([codes, mid, torch.nextafter(mid, torch.tensor(0.0)), torch.nextafter(mid, torch.tensor(1e9))])
    near = torch.cat([near, -near, torch.tensor([448.0])])
    for scale in (1.0, 0.0131, 3.7e-5, 1e-30, 2.0 ** -126 / 448, 7.3e35):
        x = (near * scale).to(DEV)
        check(dec.quantize_to_fp8(x), x, f"scale {scale}")
    for x in (torch.zeros(100), torch.full((33,), 1e-13), torch.full((17,), 1e-45), -torch.zeros(5)):
        check(dec.quantize_to_fp8(x.to(DEV)), x.to(DEV), f"{x[0].item()}")


@pytest.mark.parametrize("special", [[float("inf")], [float("-inf")], [float("nan")], [-float("nan")],
                                     [float("nan"), float("-inf"), -float("nan")]])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
def test_infinities_and_nans(special, dtype):
    x = torch.randn(5003, device=DEV).to(dtype)
    x[torch.arange(len(special), device=DEV) * 1600 + 77] = torch.tensor(special, device=DEV).to(dtype)
    x[4999] = 0
    check(dec.quantize_each_to_fp8(x)[0], x.float(), f"{special} {dtype}")


def test_three_tensors_at_once_keep_their_own_scales():
    q, k, v = (torch.randn(*s, device=DEV).bfloat16() * m for s, m in
               (((3, 32, 128), 0.3), ((3, 8, 1111, 128), 1.0), ((3, 8, 1111, 128), 40.0)))
    for got, x in zip(dec.quantize_each_to_fp8(q, k, v), (q, k, v)):
        check(got, x.float(), f"{tuple(x.shape)}")
    # a dense permuted tensor keeps its strides; a strided or unaligned one is packed
    t = k.transpose(1, 2)
    got, _ = dec.quantize_each_to_fp8(t)[0], None
    check(got, t.float(), "transposed")
    for part in (k[:, :, 5:900], k.reshape(-1)[3:5000]):
        codes, scale = dec.quantize_each_to_fp8(part)[0]
        want, ws = expression(part.float())
        assert torch.equal(scale, ws) and torch.equal(codes.view(torch.uint8), want.view(torch.uint8))


def test_lazily_negated_tensors():
    """Their memory holds the values with the other sign."""
    x = torch.randn(5003, device=DEV)
    neg = torch._neg_view(x)
    assert neg.is_neg()
    check(dec.quantize_to_fp8(neg), -x, "quantize_to_fp8")
    for t in (x, x.half(), x.bfloat16()):
        check(dec.quantize_each_to_fp8(torch._neg_view(t))[0], -t.float(), f"quantize_each_to_fp8 {t.dtype}")


def test_recorded_calls_keep_the_torch_expression():
    x = torch.randn(64, device=DEV, requires_grad=True)
    _, scale = dec.quantize_to_fp8(x)
    assert scale.grad_fn is not None
    y = torch.randn(4, 64, device=DEV)
    codes, scales = torch.func.vmap(dec.quantize_to_fp8)(y)
    for i in range(4):
        want, ws = expression(y[i])
        assert torch.equal(scales[i], ws) and torch.equal(codes[i].view(torch.uint8), want.view(torch.uint8))
