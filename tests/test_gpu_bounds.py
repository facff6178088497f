"""The attended range of an HF decode step (one launch) against the torch
operations that it replaces, over mask types, strides and row alignments."""
import pytest
import torch

from fskernels.hip import hf as H

pytest.importorskip("transformers")
pytestmark = pytest.mark.gpu
DEV = "cuda"


def both(B, S, mask=None, **kw):
    q = torch.empty(B, 4, 1, 64, dtype=torch.bfloat16, device=DEV)
    k = torch.empty(B, 2, S, 64, dtype=torch.bfloat16, device=DEV)
    got = H._decode_bounds(q, k, mask, kw)
    want = H._torch_bounds(B, S, q.device, mask if kw.get("cache_position") is None else None,
                           kw.get("cache_position"), kw.get("sliding_window"))
    for g, w in zip(got, want):
        assert (g is None) == (w is None)
        if w is not None:
            assert g.dtype == torch.int32 and torch.equal(g, w), (g, w)


def masks(ok, dtype):
    if dtype == torch.bool:
        return ok
    low = torch.finfo(dtype).min
    return torch.where(ok, torch.tensor(-0.0 if ok.shape[-1] % 2 else 0.0, dtype=dtype, device=DEV),
                       torch.tensor(low, dtype=dtype, device=DEV))


# rows shorter than, of, and around one 16-byte load, one pass of the
# workgroup's loads (256 threads x 4), and several
@pytest.mark.parametrize("S", [1, 3, 7, 8, 9, 16, 17, 31, 300, 4096, 8191, 8193, 20001])
@pytest.mark.parametrize("dtype", [torch.bool, torch.float16, torch.bfloat16, torch.float32])
def test_masks(S, dtype):
    g = torch.Generator().manual_seed(S)
    B = 9
    starts = torch.randint(0, S, (B,), generator=g)
    ends = starts + torch.randint(1, S + 1, (B,), generator=g).clamp(max=S - starts)
    starts[0], ends[0] = 0, S      # all
    ends[1] = starts[1]            # none
    starts[2], ends[2] = S - 1, S  # the last position only
    starts[3], ends[3] = 0, 1      # the first only
    at = torch.arange(S)[None]
    ok = ((at >= starts[:, None]) & (at < ends[:, None])).to(DEV)
    full = masks(ok, dtype)[:, None, None, :]
    both(B, S, full)
    both(B, S, full[:1])                                     # one row for the batch
    wide = torch.cat([full, full.flip(-1)], -1)              # a wider mask: the first S positions count
    both(B, S, wide)
    both(B, S, torch.stack([full, full.flip(0)], -1)[..., 0])  # positions two elements apart
    queries = torch.cat([full.flip(0), full], 2)             # the last query's row
    both(B, S, queries.expand(B, 3, 2, S))


def test_mask_with_gaps_and_one_column():
    ok = torch.zeros(2, 1, 1, 500, dtype=torch.bool, device=DEV)
    ok[0, ..., 40:60] = ok[0, ..., 300:333] = ok[1, ..., 499:] = True
    both(2, 500, ok)
    both(2, 77, ok[..., 40:41])  # broadcast over the positions


@pytest.mark.parametrize("window", [None, 0, 1, 100, 5000])
def test_positions_and_windows(window):
    for B in (1, 300):
        both(B, 1000, cache_position=torch.tensor([7, 411], device=DEV), sliding_window=window)
        both(B, 1000, sliding_window=window)
    both(3, 1000, cache_position=torch.arange(20, device=DEV)[::2], sliding_window=window)


def test_mask_of_another_shape_is_refused():
    for shape in ((3, 1, 1, 64), (2, 1, 1, 63), (2, 64)):
        with pytest.raises((RuntimeError, IndexError)):
            both(2, 64, torch.zeros(shape, device=DEV))
    with pytest.raises(RuntimeError):
        both(2, 64, torch.zeros(2, 1, 1, 64))
