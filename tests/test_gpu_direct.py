"""The direct kernel (one workgroup per short sequence and head) against the
float64 oracle and the split kernels, at the edges of its tiles, wave counts,
head blocks and of the rule that takes it."""
import numpy as np
import pytest
import torch

from fasterkernels_amd import native as nat
from fasterkernels_amd import workloads as W
from fskernels.hip import decode as dec
from oracle import decode_oracle as O
from tests.test_gpu_decode import assert_close, f64, oracle_for, run_and_check, tol_for

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture
def option():
    def set_option(name, value):
        nat.check(nat.load().fsk_set_option(name.encode(), value))
    yield set_option
    set_option("direct", 1)


def kernels(fn):
    """(direct kernels, partial kernels) that a call launches."""
    from torch.profiler import ProfilerActivity, profile
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        fn()
        torch.cuda.synchronize()
    names = [e.key for e in prof.key_averages()]
    return sum("direct_kernel" in n for n in names), sum("partial_kernel" in n for n in names)


def launches(wl, **kw):
    return kernels(lambda: W.run(wl, **kw))


EDGES = [1, 31, 32, 33, 64, 65, 127, 129, 255, 257, 500, 512]


@pytest.mark.parametrize("layout", ["M0", "C1"])
@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("kv", ["f16", "bf16", "e4m3"])
@pytest.mark.parametrize("longest", [32, 64, 96, 256, 384])
def test_short_sequences(layout, D, kv, longest):
    q = "f16" if kv == "f16" else "bf16"
    lens = [n for n in EDGES if n <= longest] + [longest] + [0] * 5
    Hkv = 16 if D == 256 else 4  # (head_dim 256: at least 128 workgroups beyond 64 tokens, 256 beyond 256)
    if layout == "C1" and longest > 64:
        lens = [longest // 2 - 1, 0, 1, longest // 2] + [0] * 12  # (varlen: the call's rows are the bound)
    wl = W.make(layout, overrides=dict(B=len(lens), Hq=4 * Hkv, Hkv=Hkv, D=D, kv=kv, q=q, out=q, lens=("list", lens),
                                       sinks=True), seed=D + longest)
    for mode in ("exp", "linear"):
        run_and_check(wl, mode, what=f"{layout} D={D} {kv} <= {longest} {mode}")
    assert launches(wl.to(DEV)) == (1, 0)


# one, two and four waves in many workgroups, eight in few (e4m3: in up to 256),
# the longest sequences
@pytest.mark.parametrize("kv", ["f16", "e4m3"])
@pytest.mark.parametrize("B,longest", [(300, 64), (300, 250), (300, 1024), (400, 600), (128, 896), (40, 640), (2, 250),
                                       (2, 384), (16, 512)])
def test_wave_counts(kv, B, longest):
    q = "f16" if kv == "f16" else "bf16"
    lens = [(37 * b) % (longest + 1) for b in range(B - 1)] + [longest]
    wl = W.make("M0", overrides=dict(B=B, Hq=8, Hkv=8, kv=kv, q=q, out=q, lens=("list", lens), sinks=True), seed=B)
    run_and_check(wl, what=f"{kv} {B} x {longest}")
    assert launches(wl.to(DEV)) == (1, 0)


# head blocks of 16 (one, partial, several), one query head per KV head, and
# varlen head pairs at head_dim 64 with and without a partner
@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (8, 2), (16, 2), (16, 1), (20, 1), (48, 1), (9, 3)])
@pytest.mark.parametrize("layout,D", [("M0", 128), ("C1", 64)])
def test_head_shapes(layout, D, Hq, Hkv):
    wl = W.make(layout, overrides=dict(B=3, Hq=Hq, Hkv=Hkv, D=D, lens=("list", [1, 200, 77]), sinks=True), seed=Hq)
    run_and_check(wl, what=f"{layout} Hq={Hq} Hkv={Hkv}")


@pytest.mark.parametrize("ps", [32, 64])
@pytest.mark.parametrize("kv", ["f16", "e4m3"])
def test_larger_pages_and_poisoned_entries(ps, kv):
    """Table entries past a sequence's last page are read but never used."""
    g = torch.Generator().manual_seed(ps)
    lens, Hkv, D, mb = [1, ps, ps + 1, 190], 2, 128, 256 // ps
    P = 4 * mb
    kf, vf = (torch.randn(P, Hkv, ps, D, generator=g) for _ in range(2))
    q = torch.randn(4, 8, D, generator=g).half()
    bt = torch.randperm(P, generator=g).to(torch.int32).view(4, mb).clone()
    for b, n in enumerate(lens):
        bt[b, -(-n // ps):] = torch.tensor([-1, 1 << 30, P, -(1 << 31)] * mb, dtype=torch.int64)[:mb - -(-n // ps)].to(torch.int32)
    ks = vs = None
    if kv == "e4m3":
        (kp, ks), (vp, vs) = W._quantize(kf), W._quantize(vf)
        ref = O.decode_paged(f64(q), kp.view(torch.uint8).numpy(), vp.view(torch.uint8).numpy(), bt.numpy(), lens,
                             None, "linear", float(ks), float(vs))
    else:
        kp, vp = kf.half(), vf.half()
        ref = O.decode_paged(f64(q), kp.numpy(), vp.numpy(), bt.numpy(), lens, None, "linear")
    sc = {} if ks is None else dict(k_scale=ks.to(DEV), v_scale=vs.to(DEV))
    out = dec.paged_flash_decode(q.to(DEV), kp.to(DEV), vp.to(DEV), bt.to(DEV),
                                 torch.tensor(lens, dtype=torch.int32, device=DEV), ps, **sc)
    assert_close(out, ref, *((1e-2, 0.0) if kv == "e4m3" else (2e-3, 2e-3)), f"pages of {ps} {kv}")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float8_e4m3fn])
@pytest.mark.parametrize("D", [64, 128, 256])
def test_dense_ranges(dtype, D):
    g = torch.Generator().manual_seed(D)
    S, ends, starts = 250, [250, 33, 100, 7], [0, 32, 37, 7]
    q, k, v = (torch.randn(*s, generator=g) for s in ((4, 12, D), (4, 3, S, D), (4, 3, S, D)))
    e, st = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in (ends, starts))
    if dtype == torch.float8_e4m3fn:
        (q8, sq), (k8, sk), (v8, sv) = (W._quantize(t) for t in (q, k, v))
        out = dec.flash_decode_gqa_hf_fp8(q8.to(DEV), k8.to(DEV), v8.to(DEV), e, sq.to(DEV), sk.to(DEV), sv.to(DEV),
                                          torch.float16, start_k_offsets=st)
        q, k, v = ((x8.float() * s).numpy() for x8, s in ((q8, sq), (k8, sk), (v8, sv)))
        q, tol = q.astype(np.float16), (1e-2, 0.0)
    else:
        q, k, v = (t.to(dtype) for t in (q, k, v))
        out = dec.flash_decode_gqa_hf_dense_optimized(q.to(DEV), k.to(DEV), v.to(DEV), e, st)
        q, k, v, tol = *(f64(t) for t in (q, k, v)), (2e-3, 2e-3)
    ref = O.decode_dense(np.asarray(q, np.float64), np.asarray(k, np.float64), np.asarray(v, np.float64), ends, starts)
    assert_close(out[:3], ref[:3], *tol, f"dense {dtype} D={D}")
    assert torch.isnan(out[3]).all()  # an empty range without a sink: 0 / 0


@pytest.mark.parametrize("out", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("layout", ["M0", "C1"])
@pytest.mark.parametrize("mode", ["exp", "linear"])
def test_block_scores(layout, out, mode, option):
    lens = [1, 127, 128, 129, 0, 257, 384] if layout == "M0" else [1, 200, 0, 130]
    wl = W.make(layout, overrides=dict(B=len(lens), Hq=36, Hkv=2, lens=("list", lens), sinks=True, out=out),
                seed=3).to(DEV)
    assert launches(wl, block_scores=True) == (1, 0)
    got, scores = W.run(wl, sink_mode=mode, block_scores=True)
    option("direct", 0)
    assert launches(wl, block_scores=True) == (0, 1)
    want, want_scores = W.run(wl, sink_mode=mode, block_scores=True)
    for a, b in ((got, want), (scores, want_scores)):
        assert a.dtype == b.dtype and a.shape == b.shape
        # both within a rounding of the exact value (P is rounded alike; outputs differ by the sums' order)
        assert_close(a, f64(b), 1e-3, 8e-3 if out == "bf16" else 1e-3, "direct and split")
    assert (f64(scores)[lens.index(0)] == 0).all()
    assert torch.equal(scores == 0, want_scores == 0)


# (query heads, batch, longest sequence, direct): both sides of the rule's lines
# for 8 KV heads x 128: fp16 by K/V bytes of a head, e4m3 by tokens
@pytest.mark.parametrize("kv,Hq,B,longest,direct", [
    ("f16", 32, 1, 384, 1), ("f16", 32, 1, 385, 0), ("f16", 32, 15, 384, 1), ("f16", 32, 15, 1024, 0),
    ("f16", 32, 16, 640, 1), ("f16", 32, 16, 641, 0), ("f16", 32, 32, 768, 1), ("f16", 32, 32, 769, 0),
    ("f16", 32, 48, 640, 1), ("f16", 32, 48, 641, 0), ("f16", 32, 51, 768, 1), ("f16", 32, 64, 896, 1),
    ("f16", 32, 64, 897, 0), ("f16", 32, 96, 1024, 1), ("f16", 32, 96, 1025, 0),
    ("f16", 8, 16, 512, 1), ("f16", 8, 16, 513, 0), ("f16", 8, 192, 1024, 1), ("f16", 8, 191, 1024, 0),
    ("f16", 32, 300, 100, 1), ("e4m3", 32, 1, 768, 1), ("e4m3", 32, 2, 769, 0), ("e4m3", 32, 20, 896, 1),
    ("e4m3", 32, 20, 897, 0), ("e4m3", 32, 32, 1024, 1), ("e4m3", 32, 32, 1025, 0)])
def test_rule(kv, Hq, B, longest, direct, option):
    lens = [(7 * b) % longest + 1 for b in range(B - 1)] + [longest]
    q = "f16" if kv == "f16" else "bf16"
    wl = W.make("M0", overrides=dict(B=B, Hq=Hq, lens=("list", lens), kv=kv, q=q, out=q), seed=B)
    run_and_check(wl, what=f"{kv} Hq={Hq} {B} x {longest}")
    wl = wl.to(DEV)
    assert launches(wl) == (direct, 1 - direct)
    assert launches(wl, chunk_tokens=64) == (0, 1)  # a fixed split is the split kernels'
    host = W.run(wl, host_lengths=True) if B <= 64 else None
    if host is not None:
        assert torch.equal(host, W.run(wl))
    option("direct", 0)
    assert launches(wl) == (0, 1)


# a split-count hint makes every full-length sequence split: chunks of at most
# ceil(S / n) tokens, rounded up to 32, keep the split kernels where that is
# less than S
@pytest.mark.parametrize("S,splits,direct", [(384, 1, 1), (384, 2, 0), (384, 8, 0), (64, 2, 0), (33, 2, 0), (32, 8, 1)])
def test_split_hints_keep_the_split_kernels(S, splits, direct):
    g = torch.Generator().manual_seed(S)
    q, k, v = (torch.randn(*s, generator=g).half() for s in ((2, 8, 128), (2, 2, S, 128), (2, 2, S, 128)))
    lens = torch.tensor([S, S - 5], dtype=torch.int32, device=DEV)
    args = q.to(DEV), k.to(DEV), v.to(DEV), lens
    (q8, sq), (k8, sk), (v8, sv) = (W._quantize(t.float()) for t in (q, k, v))
    args8 = (q8.to(DEV), k8.to(DEV), v8.to(DEV), lens, sq.to(DEV), sk.to(DEV), sv.to(DEV), torch.float16)
    ref = O.decode_dense(f64(q), f64(k), f64(v), lens.cpu().numpy(), None)
    dec.set_num_splits_fp8(splits)
    try:
        assert kernels(lambda: dec.flash_decode_gqa_hf_fp8(*args8)) == (direct, 1 - direct)
    finally:
        dec.set_num_splits_fp8(1)
    assert kernels(lambda: dec.flash_decode_gqa_hf_dense_optimized(*args, num_splits=splits)) == (direct, 1 - direct)
    dec.set_num_splits(splits)
    try:
        assert kernels(lambda: dec.flash_decode_gqa_hf_dense_optimized(*args)) == (direct, 1 - direct)
        assert_close(dec.flash_decode_gqa_hf_dense_optimized(*args), ref, 2e-3, 2e-3, f"S={S} splits={splits}")
    finally:
        dec.set_num_splits(1)


def test_captured_and_replayed():
    wl = W.make("M0", overrides=dict(B=5, lens=("list", [3, 100, 256, 31, 64])), seed=1).to(DEV)
    from fskernels.engine.hip_graph import DecodeGraph
    step = DecodeGraph(W.run, wl)
    for seed in range(4):
        wl.q.copy_(torch.randn(wl.q.shape, generator=torch.Generator().manual_seed(seed)).half())
        wl.seq_lens.copy_(torch.tensor([(3 + 50 * seed) % 256 + 1, 100, 256 - seed, 31, 64], dtype=torch.int32))
        got = step.replay().clone()
        torch.cuda.synchronize()
        assert torch.equal(got, W.run(wl))
