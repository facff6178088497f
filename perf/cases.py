"""Cases that time the decode-attention path over the range that it is used in.

One case is one call (or one layer's step) of the public entry points: paged
decode over a block table (continuous batching), varlen decode with attention
sinks, decode over a dense HF cache (fp16/bf16 and e4m3), the HF attention
functions with the mask they are handed, the KV write of a prefill into
scattered pages, and the per-layer step of a serving loop (store one new row
per sequence, then attend).  Sizes are those of the benchmark configurations
and tests of this repository, or between them.

Sequence lengths come from the case alone (its ``length_seed``), so that the
work of a case is known; values, page tables, masks' positions and scales come
from the seed that ``prepare`` is given.
"""
from __future__ import annotations

import math
import random

import torch

PAGE = 16
DT = {"f16": torch.float16, "bf16": torch.bfloat16, "e4m3": torch.float8_e4m3fn, "f32": torch.float32}
SIZE = {"f16": 2, "bf16": 2, "e4m3": 1, "f32": 4}

# (query heads, KV heads, head_dim): the benchmark's and the tests' head shapes
HEADS = [(32, 8, 128), (64, 8, 128), (16, 8, 128), (8, 8, 128), (40, 8, 128), (32, 4, 128), (64, 4, 128),
         (32, 1, 128), (64, 8, 64), (32, 8, 64), (32, 8, 256), (16, 8, 256)]


def _case(kind, batch, heads, kv, dist, lo, hi, length_seed, *, sinks="none", name=None):
    hq, hkv, d = heads
    c = dict(kind=kind, batch=batch, q_heads=hq, kv_heads=hkv, head_dim=d, kv=kv, dist=dist, lo=lo, hi=hi,
             length_seed=length_seed, sinks=sinks)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # One conversation just begun: the smallest decode call, all latency and launches.
        _case("paged", 1, (32, 8, 128), "f16", "uniform", 517, 517, 1, name="paged_one_short"),
        # A full server: 32 sequences of 1K-16K tokens on shuffled pages (the largest case).
        _case("paged", 32, (32, 8, 128), "f16", "uniform", 1024, 16384, 103, name="paged_ragged"),
        # A chat server with many short conversations, pools in the type that PagedKVCache.from_config gives them.
        _case("paged", 256, (32, 8, 128), "bf16", "uniform", 16, 1024, 3, name="paged_many_short"),
        # e4m3 pools with per-tensor scales, bf16 queries, sinks, lognormal lengths (long-tailed traffic).
        _case("paged", 64, (32, 8, 128), "e4m3", "lognormal", 16, 32768, 105, sinks="exp", name="paged_e4m3_sinks"),
        # Decode that also returns the pooled block scores (sparse-attention block selection).
        _case("scores", 4, (32, 8, 128), "f16", "uniform", 4096, 16384, 5, sinks="linear", name="paged_scores"),
        # The reference benchmark's varlen decode, a middle point of its sweep.
        _case("varlen", 4, (32, 8, 128), "f16", "uniform", 1024, 4096, 42, sinks="linear", name="varlen_sinks"),
        # head_dim 64 with sink logits and eight queries per KV head, packed rows of odd lengths.
        _case("varlen", 8, (64, 8, 64), "bf16", "lognormal", 16, 32768, 106, sinks="exp", name="varlen_d64_sinks"),
        # An HF model's decode step on a left-padded batch in a static cache, through the attention function.
        _case("hf", 4, (32, 8, 128), "bf16", "uniform", 700, 2048, 8, name="hf_attention"),
        # The same hook with fp8: Q, K and V quantised on every call, as the reference's patch does.
        _case("hf_fp8", 4, (32, 8, 128), "bf16", "uniform", 1500, 4096, 9, name="hf_attention_fp8"),
        # A dense e4m3 cache that was quantised once, e4m3 queries, ragged ends.
        _case("dense_fp8", 8, (32, 8, 128), "e4m3", "uniform", 500, 8191, 10, name="dense_e4m3"),
        # One layer of a serving loop's step: the new rows stored, then the batch attends.
        _case("step", 24, (32, 8, 128), "bf16", "uniform", 100, 3000, 11, name="layer_step"),
        # A prefill's rows quantised into a fragmented e4m3 pool.
        _case("write", 8, (32, 8, 128), "e4m3", "uniform", 2000, 6000, 12, name="kv_prefill_e4m3"),
    ]


KINDS = ["paged", "paged", "paged", "varlen", "varlen", "scores", "hf", "hf_fp8", "dense_fp8", "step", "write", "write"]
# Tokens of one call, over all its sequences: from one short sequence to the largest listed case.
MOST_TOKENS = {"paged": 270000, "varlen": 270000, "scores": 130000, "hf": 64000, "hf_fp8": 14000,
               "dense_fp8": 100000, "step": 130000, "write": 33000}


def draw(rng: random.Random):
    """A case of the same ranges: any kind, sizes spread over their logarithms."""
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(KINDS)
    heads = rng.choice(HEADS)
    kv = {"hf": rng.choice(["bf16", "f16"]), "hf_fp8": rng.choice(["bf16", "f16"]), "dense_fp8": "e4m3"}.get(
        kind, rng.choice(["f16", "bf16", "e4m3"]))
    # the same K/V bytes per token as 8 heads of 128 allow the same number of tokens
    most = int(MOST_TOKENS[kind] * 1024 / max(heads[1] * heads[2], 1024))
    batch = log_int(1, {"hf": 16, "hf_fp8": 8, "dense_fp8": 32, "write": 16}.get(kind, 512))
    top = max(33, min(32768, most // batch))
    hi = log_int(32, top)
    dist = rng.choice(["uniform", "uniform", "lognormal"])
    lo = hi if rng.random() < 0.2 else rng.randint(1, hi) if dist == "uniform" else 1
    sinks = rng.choice(["none", "linear", "exp"]) if kind in ("paged", "varlen", "scores") else "none"
    return _case(kind, batch, heads, kv, dist, lo, hi, rng.randrange(1 << 30), sinks=sinks)


def _lengths(c):
    """The case's sequence lengths, from the case alone."""
    r = random.Random(c["length_seed"])
    lo, hi = c["lo"], c["hi"]
    if c["dist"] == "uniform":
        return [r.randint(lo, hi) for _ in range(c["batch"])]
    # long-tailed: the mode near an eighth of the longest
    mu = math.log(max(hi / 8.0, 1.0))
    return [int(min(max(round(math.exp(r.gauss(mu, 1.0))), lo), hi)) for _ in range(c["batch"])]


def _quantize(x):
    """e4m3 codes and the per-tensor scale of fp32 values, as the path's callers make them once."""
    scale = x.abs().max().clamp(min=1e-12) / 448.0
    return (x / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn), scale


def _store(x, kv):
    return _quantize(x) if kv == "e4m3" else (x.to(DT[kv]), None)


def _inputs(c, seed):
    """Q, K, V and tables on the GPU, from the seed alone."""
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    B, Hq, Hkv, D, kv = c["batch"], c["q_heads"], c["kv_heads"], c["head_dim"], c["kv"]
    lens = _lengths(c)
    kind = c["kind"]
    s = dict(case=c, lens=lens)

    def randn(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    if kind in ("paged", "scores", "step", "write"):
        npages = [-(-n // PAGE) for n in lens]
        total = sum(npages)
        P = total + total // 10 + 1
        perm = torch.randperm(P, generator=g, device=dev).to(torch.int32)
        table = torch.full((B, max(npages)), -1, dtype=torch.int32)
        host = perm.cpu()
        off = 0
        for b, n in enumerate(npages):
            table[b, :n] = host[off:off + n]
            off += n
        s["table"] = table.to(dev)
        s["lens_dev"] = torch.tensor(lens, dtype=torch.int32, device=dev)
        shape = (P, Hkv, PAGE, D)
    elif kind == "varlen":
        cu = torch.zeros(B + 1, dtype=torch.int32)
        cu[1:] = torch.cumsum(torch.tensor(lens), 0).to(torch.int32)
        s["cu"] = cu.to(dev)
        shape = (sum(lens), Hkv, D)
    else:
        shape = (B, Hkv, max(lens), D)

    if kind == "write":
        # the prompt's new rows, sequence after sequence, and where they go
        n = sum(lens)
        src = "bf16" if kv == "e4m3" else kv
        s["k_new"], s["v_new"] = randn(n, Hkv, D).to(DT[src]), randn(n, Hkv, D).to(DT[src])
        at = torch.cat([torch.arange(m) for m in lens])
        row = torch.repeat_interleave(torch.arange(B), torch.tensor(lens))
        s["slots"] = (table[row, at // PAGE].long() * PAGE + at % PAGE).to(dev)
        s["k"] = torch.zeros(shape, dtype=torch.uint8 if kv == "e4m3" else DT[kv], device=dev).view(DT[kv])
        s["v"] = torch.zeros_like(s["k"])
        s["k_scale"] = s["v_scale"] = None
        if kv == "e4m3":
            s["k_scale"] = torch.tensor(0.011, device=dev)
            s["v_scale"] = torch.tensor(0.009, device=dev)
        return s

    s["k"], s["k_scale"] = _store(randn(*shape), kv)
    s["v"], s["v_scale"] = _store(randn(*shape), kv)
    q = randn(B, Hq, D)
    s["q_scale"] = None
    if kind == "dense_fp8":
        s["q"], s["q_scale"] = _quantize(q)
    else:
        s["q"] = q.to(DT["bf16" if kv == "e4m3" else kv])
    s["sinks"] = None
    if c["sinks"] != "none":
        s["sinks"] = randn(Hq) * (0.1 if c["sinks"] == "linear" else 1.0)
    if kind in ("hf", "hf_fp8"):
        # left-padded batch: sequence b attends the last lens[b] of the positions filled so far
        S = shape[2]
        start = torch.tensor([S - n for n in lens], device=dev)
        ok = torch.arange(S, device=dev)[None] >= start[:, None]
        low = torch.finfo(s["q"].dtype).min
        s["mask"] = torch.zeros(B, 1, 1, S, dtype=s["q"].dtype, device=dev).masked_fill(~ok[:, None, None], low)
        s["q"] = s["q"].view(B, Hq, 1, D)
    if kind == "dense_fp8":
        s["lens_dev"] = torch.tensor(lens, dtype=torch.int32, device=dev)
    if kind == "step":
        # each sequence's newest row goes to its last position
        src = "bf16" if kv == "e4m3" else kv
        s["k_new"], s["v_new"] = randn(B, Hkv, D).to(DT[src]), randn(B, Hkv, D).to(DT[src])
        last = torch.tensor(lens) - 1
        s["slots"] = (table[torch.arange(B), last // PAGE].long() * PAGE + last % PAGE).to(dev)
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    from fskernels.hip import decode, kv_write  # noqa: F401  (the entry points that run() calls)
    s["decode"], s["write"] = decode, kv_write.paged_kv_write
    if case["kind"] in ("hf", "hf_fp8"):
        from fskernels.hip import hf
        s["hf"] = hf.custom_hf_decode_attention_forward_fp8 if case["kind"] == "hf_fp8" else \
            hf.custom_hf_decode_attention_forward
    return s


def run(s):
    c, kind, d = s["case"], s["case"]["kind"], s["decode"]
    mode = "exp" if c["sinks"] == "exp" else "linear"
    if kind == "paged":
        return d.paged_flash_decode(s["q"], s["k"], s["v"], s["table"], s["lens_dev"], PAGE, s_aux=s["sinks"],
                                    k_scale=s["k_scale"], v_scale=s["v_scale"], sink_mode=mode)
    if kind == "scores":
        return d.paged_flash_decode(s["q"], s["k"], s["v"], s["table"], s["lens_dev"], PAGE, s_aux=s["sinks"],
                                    k_scale=s["k_scale"], v_scale=s["v_scale"], sink_mode=mode,
                                    return_block_scores=True)
    if kind == "varlen":
        return d.flash_decode_gqa_varlen(s["q"], s["k"], s["v"], s["cu"], s["sinks"], k_scale=s["k_scale"],
                                         v_scale=s["v_scale"], sink_mode=mode)
    if kind == "dense_fp8":
        return d.flash_decode_gqa_hf_fp8(s["q"], s["k"], s["v"], s["lens_dev"], s["q_scale"], s["k_scale"],
                                         s["v_scale"], torch.bfloat16)
    if kind in ("hf", "hf_fp8"):
        return s["hf"](None, s["q"], s["k"], s["v"], s["mask"], c["head_dim"] ** -0.5)[0]
    s["write"](s["k_new"], s["v_new"], s["k"], s["v"], s["slots"], k_scale=s["k_scale"], v_scale=s["v_scale"])
    pools = (s["k"].view(torch.uint8), s["v"].view(torch.uint8)) if c["kv"] == "e4m3" else (s["k"], s["v"])
    if kind == "write":
        return pools
    out = d.paged_flash_decode(s["q"], s["k"], s["v"], s["table"], s["lens_dev"], PAGE, k_scale=s["k_scale"],
                               v_scale=s["v_scale"])
    return (out, *pools)


def work(case):
    B, Hq, Hkv, D, kind = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"], case["kind"]
    lens = _lengths(case)
    n = sum(lens)
    e = SIZE[case["kv"]]
    src = 2 if case["kv"] == "e4m3" else e
    if kind == "write":
        return {"bytes": n * (Hkv * D * 2 * (src + e) + 8), "flops": 0}
    flops = 4 * D * Hq * n
    nbytes = n * Hkv * D * 2 * e + B * Hq * D * (2 if kind != "dense_fp8" else 1) + B * Hq * D * 2 + 4 * B
    if kind in ("paged", "scores", "step"):
        nbytes += 4 * sum(-(-m // PAGE) for m in lens)
    if kind == "scores":
        nbytes += B * Hq * 2 * (-(-(-(-max(lens) // PAGE) * PAGE) // 128))
    if kind == "step":
        nbytes += B * (Hkv * D * 2 * (src + e) + 8)
    if kind in ("hf", "hf_fp8"):
        nbytes += B * max(lens) * 2
    if kind == "hf_fp8":
        # the scales are of the whole tensors, padding included
        nbytes += (B * max(lens) - n) * Hkv * D * 2 * e
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times what the kernels show against ``exact`` (rel 2.5e-4 to
    2.8e-4 with fp16 results, 1.6e-3 to 1.7e-3 with bf16 ones): the final
    rounding to the output type and, under it, P rounded to the value type.
    Stored rows and codes are the same bytes."""
    if case["kind"] == "write":
        return "exact"
    if case["kv"] != "f16":
        return {"rel": 7e-3, "max": 2e-2}
    # fp8 through the HF function: Q is rounded to fp16 once more
    return {"rel": 2e-3, "max": 1e-2} if case["kind"] == "hf_fp8" else {"rel": 1.1e-3, "max": 5e-3}


def _attend(q, k, v, scale, sink, mode):
    """One sequence in 64 bits: q [Hq, D], k / v [Hkv, n, D]; also the probabilities."""
    hkv = k.shape[0]
    qg = q.view(hkv, -1, q.shape[-1])
    x = torch.matmul(qg, k.transpose(1, 2).contiguous()).reshape(q.shape[0], -1) * scale
    m = x.amax(-1, keepdim=True)
    p = torch.exp(x - m)
    den = p.sum(-1, keepdim=True)
    if sink is not None:
        z = sink.double()[:, None]
        den = den + (torch.exp(z - m) if mode == "exp" else z)
    p = p / den
    return torch.matmul(p.view(hkv, -1, p.shape[-1]), v).reshape(q.shape), p


def exact(case, seed):
    s = _inputs(case, seed)
    c, kind, lens = case, case["kind"], s["lens"]
    mode = "exp" if c["sinks"] == "exp" else "linear"
    Hq, D = c["q_heads"], c["head_dim"]
    if kind in ("write", "step"):
        page, row = s["slots"] // PAGE, s["slots"] % PAGE
        for pool, new, sc in ((s["k"], s["k_new"], s["k_scale"]), (s["v"], s["v_new"], s["v_scale"])):
            if c["kv"] == "e4m3":
                codes = (new.float() / sc).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
                pool.view(torch.uint8)[page, :, row, :] = codes.view(torch.uint8)
            else:
                pool[page, :, row, :] = new
        pools = (s["k"].view(torch.uint8), s["v"].view(torch.uint8)) if c["kv"] == "e4m3" else \
            (s["k"].double(), s["v"].double())
        if kind == "write":
            return pools
    q, k, v = s["q"], s["k"], s["v"]
    ks, vs = s["k_scale"], s["v_scale"]
    qs = s["q_scale"]
    if kind == "hf_fp8":
        (q, qs), (k, ks), (v, vs) = (_quantize(t.float()) for t in (q, k, v))
    q = q.double() * (1.0 if qs is None else qs.double())
    out = torch.empty(c["batch"], Hq, D, dtype=torch.float64, device=q.device)
    n_blk = -(-(max(-(-n // PAGE) for n in lens) * PAGE) // 128)
    blocks = torch.zeros(c["batch"], Hq, n_blk, dtype=torch.float64, device=q.device)
    at = 0
    for b, n in enumerate(lens):
        if kind in ("paged", "scores", "step"):
            pages = s["table"][b, :-(-n // PAGE)].long()
            kb, vb = (t[pages].transpose(0, 1).reshape(c["kv_heads"], -1, D)[:, :n] for t in (k, v))
        elif kind == "varlen":
            kb, vb = (t[at:at + n].transpose(0, 1) for t in (k, v))
            at += n
        elif kind == "dense_fp8":
            kb, vb = k[b, :, :n], v[b, :, :n]
        else:
            kb, vb = k[b, :, max(lens) - n:], v[b, :, max(lens) - n:]
        kb = kb.double().contiguous() * (1.0 if ks is None else ks.double())
        vb = vb.double().contiguous() * (1.0 if vs is None else vs.double())
        out[b], p = _attend(q[b].reshape(Hq, D), kb, vb, D ** -0.5, s["sinks"], mode)
        if kind == "scores":
            m = -(-n // 128)
            pad = torch.zeros(Hq, m * 128, dtype=torch.float64, device=q.device)
            pad[:, :n] = p
            blocks[b, :, :m] = pad.view(Hq, m, 128).amax(-1)
    if kind == "scores":
        return out, blocks
    return (out, *pools) if kind == "step" else out
