"""The fp8 attention hook's quantising decode against the same call in three
steps: the range, the stored codes (bit-exact with the torch expression,
tests/test_gpu_quantize.py) and the decode of them."""
import pytest
import torch

pytest.importorskip("transformers")

from fasterkernels_amd import native as nat  # noqa: E402
from fskernels.hip import decode as dec  # noqa: E402
from fskernels.hip import hf as H  # noqa: E402
from tests.test_gpu_decode import assert_close, f64  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda"


def steps(q, k, v, mask, scaling, **kw):
    lens, starts = H._decode_bounds(q, k, mask, kw)
    (q8, sq), (k8, sk), (v8, sv) = dec.quantize_each_to_fp8(q.squeeze(2), k, v)
    return dec.flash_decode_gqa_hf_fp8(q8, k8, v8, lens, sq, sk, sv, q.dtype, start_k_offsets=starts,
                                       sm_scale=scaling)


def inputs(B, Hq, Hkv, S, D, dtype, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(B, Hq, 1, D, generator=g, device=DEV).to(dtype),
            torch.randn(B, Hkv, S, D, generator=g, device=DEV).to(dtype) * 1.7,
            torch.randn(B, Hkv, S, D, generator=g, device=DEV).to(dtype) * 0.3)


def padding_mask(B, S, dtype, seed=0):
    g = torch.Generator().manual_seed(seed)
    start = torch.randint(0, S, (B,), generator=g).to(DEV)
    hidden = torch.arange(S, device=DEV)[None] < start[:, None]
    if B > 1:
        hidden[1] = True
        hidden[1, S // 2] = False
    return torch.zeros(B, 1, 1, S, dtype=dtype, device=DEV).masked_fill(hidden[:, None, None], torch.finfo(dtype).min)


def check(q, k, v, mask, what, **kw):
    scaling = 0.7 * q.shape[-1] ** -0.5
    out, _ = H.custom_hf_decode_attention_forward_fp8(None, q, k, v, mask, scaling, **kw)
    want = steps(q, k, v, mask, scaling, **kw)
    assert out.dtype == want.dtype and out.shape == want.shape
    # The same codes and scales; where one of the two takes the direct kernel
    # the sums' order differs, and with it P's rounding to f16 (2^-11 of values
    # up to ~1.3) and the output's own.
    ulp = 2.0 ** -7 if q.dtype == torch.bfloat16 else 2.0 ** -9
    assert_close(out, f64(want), 1e-3, ulp, what)


# short ranges (the direct kernel), one split and many, tiles' edges
@pytest.mark.parametrize("S", [1, 31, 33, 200, 700, 5000])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_matches_the_three_steps(S, D, dtype):
    q, k, v = inputs(3, 16, 4, S, D, dtype, seed=S + D)
    check(q, k, v, padding_mask(3, S, dtype), f"S={S} D={D} {dtype}")
    check(q, k, v, None, f"S={S} D={D} {dtype} no mask")


# The split kernels quantising on the way give the very result of the stored
# codes' decode: the split, the tiles and every sum's order are the same.
@pytest.mark.parametrize("S,Hq,Hkv", [(1, 16, 4), (33, 16, 4), (700, 6, 2), (5000, 16, 4), (16000, 32, 2)])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_split_results_are_those_of_the_stored_codes(S, Hq, Hkv, D, dtype):
    q, k, v = inputs(3, Hq, Hkv, S, D, dtype, seed=S + D)
    mask, scaling = padding_mask(3, S, dtype), 0.7 * D ** -0.5
    nat.set_option("direct", 0)
    try:
        for m in (mask, None):
            out, _ = H.custom_hf_decode_attention_forward_fp8(None, q, k, v, m, scaling)
            assert torch.equal(out, steps(q, k, v, m, scaling)), f"S={S} D={D} {dtype} mask={m is not None}"
    finally:
        nat.set_option("direct", 1)


@pytest.mark.parametrize("Hq,Hkv", [(8, 8), (64, 4), (3, 1), (40, 2)])
def test_head_shapes(Hq, Hkv):
    """(40, 2): 20 query heads per KV head take the stored codes."""
    q, k, v = inputs(2, Hq, Hkv, 600, 128, torch.bfloat16, seed=Hq)
    check(q, k, v, padding_mask(2, 600, torch.bfloat16), f"Hq={Hq} Hkv={Hkv}")


def test_positions_windows_and_hints():
    q, k, v = inputs(2, 16, 8, 3000, 128, torch.bfloat16)
    at = torch.tensor([7, 2222], device=DEV)
    check(q, k, v, None, "position", cache_position=at)
    check(q, k, v, None, "position and window", cache_position=at, sliding_window=100)
    check(q, k, v, None, "window", sliding_window=1000)
    dec.set_num_splits_fp8(8)
    try:
        check(q, k, v, None, "split hint", cache_position=at)
    finally:
        dec.set_num_splits_fp8(1)


def test_strides():
    """Views with gaps, permuted heads, contiguous tensors that do not start
    16-byte aligned and rows of an odd stride; a cache with more sequences than
    the batch (its scales cover all of them)."""
    q, k, v = inputs(4, 16, 4, 520, 128, torch.bfloat16)
    check(q, k[:, :, 3:400], v[:, :, 3:400], None, "gaps")
    check(q.transpose(0, 1).contiguous().transpose(0, 1), k.transpose(1, 2).contiguous().transpose(1, 2),
          v.transpose(1, 2).contiguous().transpose(1, 2), None, "permuted")
    for at in range(3):
        t = [q, k, v]
        off = torch.empty(t[at].numel() + 8, dtype=q.dtype, device=DEV)
        t[at] = off[3:3 + t[at].numel()].view(t[at].shape).copy_(t[at])
        assert t[at].is_contiguous() and t[at].data_ptr() % 16
        check(*t, None, f"tensor {at} at an odd offset")
        wide = torch.empty(*[q, k, v][at].shape[:-1], 131, dtype=q.dtype, device=DEV)
        t[at] = wide[..., :128].copy_([q, k, v][at])
        check(*t, None, f"tensor {at} with rows of 131")
    k[3] *= 5
    check(q[:2], k, v, None, "more sequences than the batch")
    check(q, k[:1].expand(4, -1, -1, -1), v, None, "expanded")


def test_lazily_negated_tensors():
    """Their memory holds the values with the other sign: the call on views is
    the call on the values."""
    t = inputs(2, 8, 2, 300, 128, torch.float16)
    want, _ = H.custom_hf_decode_attention_forward_fp8(None, -t[0], t[1], -t[2], None, 0.1)
    got, _ = H.custom_hf_decode_attention_forward_fp8(None, torch._neg_view(t[0]), t[1], torch._neg_view(t[2]), None, 0.1)
    assert torch.equal(got, want)


# One special value in K, V or Q reaches every scale's codes as torch's max and
# casts carry it: the same elements come out NaN.
@pytest.mark.parametrize("which", [0, 1, 2])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 0.0])
def test_special_values(which, value):
    t = inputs(2, 8, 2, 300, 128, torch.float16)
    if value == 0.0:
        t[which].zero_()
    else:
        t[which].view(-1)[77] = value
    check(*t, None, f"{which} {value}")
