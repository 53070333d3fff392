"""The attention work a serving program has this library do, as cases that can be timed.

A case is a plain dict; ``prepare`` makes what such a program holds on the GPU before the call
(queries, paged K/V pools, block tables, lengths, new rows), ``run`` is one pass through the
public entry points, ``work`` the bytes and operations the pass cannot do without and ``exact``
the same results in 64 bits with plain torch.

Kinds of cases:
  * ``decode``: one query token per sequence over the cache (``paged_gqa_decode``), on bf16 or
    fp8 caches, uniform, log-uniform (ragged) and fixed lengths;
  * ``step``: the serving loop's decode step, which appends the sequence's newest token and
    attends in one call (``BoundDecodeAppend``);
  * ``extend``: several new tokens per sequence, causal (``paged_gqa_decode_append``): the
    verification of a few draft tokens, a chunk of a long prompt over the context already
    cached, or a whole prompt into an empty cache;
  * ``shard``: one GPU's part of a decode whose keys are spread over several GPUs: the partial
    decode of its own keys, then the merge of every GPU's gathered partials.
"""

from __future__ import annotations

import math
import random

import torch

import mx_flash_attn_kernel_opt__amd as mx

GEN_CHUNK = 1 << 25


def listed():
    return [
        # A small chat batch: a call of a few microseconds, where launch and host work count.
        dict(name="decode_tiny", kind="decode", batch=4, hq=32, hkv=8, d=128, page=16,
             lens="uniform", lo=64, hi=512, fp8=False),
        # Llama-3-8B's shape, 64 sequences of 4 096 tokens: the usual large decode batch.
        dict(name="decode_llama3_8b", kind="decode", batch=64, hq=32, hkv=8, d=128, page=16,
             lens="uniform", lo=4096, hi=4096, fp8=False),
        # Continuous batching: 256 sequences of every age, a group of 7, pages of 64.
        dict(name="decode_ragged", kind="decode", batch=256, hq=28, hkv=4, d=128, page=64,
             lens="ragged", lo=1, hi=8192, fp8=False),
        # One long document: few units of work, so the keys have to be split.
        dict(name="decode_long_b1", kind="decode", batch=1, hq=64, hkv=8, d=128, page=16,
             lens="uniform", lo=32768, hi=32768, fp8=False),
        # Large head dim, two KV heads.
        dict(name="decode_d256", kind="decode", batch=64, hq=16, hkv=2, d=256, page=16,
             lens="uniform", lo=4096, hi=8192, fp8=False),
        # An fp8 cache, lengths as a running batch has them.
        dict(name="decode_fp8", kind="decode", batch=64, hq=32, hkv=8, d=128, page=16,
             lens="uniform", lo=1024, hi=8192, fp8=True),
        # The serving loop's step with small heads: append one token, attend.
        dict(name="step_d64", kind="step", batch=128, hq=32, hkv=4, d=64, page=16,
             lens="uniform", lo=512, hi=8191, new=1, fp8=False),
        # Speculative decoding: 8 draft tokens of each of 64 sequences verified in one call.
        dict(name="verify8", kind="extend", batch=64, hq=32, hkv=8, d=128, page=16,
             lens="uniform", lo=1024, hi=4088, new=8, fp8=False),
        # Four whole prompts of 1 500 tokens into an empty cache.
        dict(name="prompt_b4", kind="extend", batch=4, hq=32, hkv=8, d=128, page=16,
             lens="uniform", lo=0, hi=0, new=1500, fp8=False),
        # A 512-token chunk of a long prompt over 16K cached tokens.
        dict(name="chunk_b1_16k", kind="extend", batch=1, hq=32, hkv=8, d=128, page=16,
             lens="uniform", lo=16384, hi=16384, new=512, fp8=False),
        # Prompt chunks of two sequences into an fp8 cache, a group of 7.
        dict(name="chunk_fp8", kind="extend", batch=2, hq=28, hkv=4, d=128, page=64,
             lens="uniform", lo=2000, hi=6000, new=1024, fp8=True),
        # One GPU's quarter of four 64K-token sequences, then the merge of the four partials.
        dict(name="shard_b4", kind="shard", batch=4, hq=64, hkv=8, d=128, page=16,
             lens="uniform", lo=16000, hi=16384, parts=4, fp8=False),
    ]


# Most K/V bytes and operations of a drawn case: the largest listed decode and prompt chunk.
MAX_KV_BYTES = 1 << 30
MAX_FLOPS = 1.2e11

# (query heads, KV heads, head dim): the shapes of the listed cases, MHA and MQA among them.
HEADS = [(32, 8, 128), (64, 8, 128), (28, 4, 128), (32, 4, 64), (16, 2, 256), (8, 8, 128),
         (32, 1, 128)]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random):
    kind = rng.choice(["decode", "decode", "decode", "step", "verify", "chunk", "chunk",
                       "prompt", "shard"])
    hq, hkv, d = rng.choice(HEADS)
    case = dict(kind=kind, batch=1, hq=hq, hkv=hkv, d=d, page=rng.choice([16, 16, 32, 64, 256]),
                lens="uniform", lo=1, hi=1, fp8=kind != "shard" and rng.random() < 0.3)
    if kind in ("decode", "step", "verify", "shard"):
        case["hi"] = _log_int(rng, 64, 65536)
        case["lo"] = rng.choice([1, case["hi"] // 2, case["hi"]])
        case["lens"] = rng.choice(["uniform", "ragged"])
        case["batch"] = _log_int(rng, 1, 16 if kind == "shard" else 256)
        if kind == "step":
            case["new"] = 1
        elif kind == "verify":
            case.update(kind="extend", new=rng.randint(2, 16))
        elif kind == "shard":
            case["parts"] = rng.randint(2, 8)
    else:
        case.update(kind="extend", new=_log_int(rng, 48, 2048), batch=_log_int(rng, 1, 8))
        case["hi"] = 0 if kind == "prompt" else _log_int(rng, 128, 32768)
        case["lo"] = rng.choice([0, case["hi"]])
    # No more than the largest listed case: fewer sequences, then shorter ones.
    while _token_bytes(case) * case["batch"] * case["hi"] > MAX_KV_BYTES or \
            _flops(case, [case["hi"]] * case["batch"]) > MAX_FLOPS:
        if case["batch"] > 1:
            case["batch"] = max(1, case["batch"] * 3 // 4)
        elif case["hi"] > 64:
            case["hi"] = case["hi"] * 3 // 4
            case["lo"] = min(case["lo"], case["hi"])
        else:
            case["new"] = case["new"] * 3 // 4
    return case


def _token_bytes(case) -> int:
    """K and V bytes of one cached token."""
    return 2 * case["hkv"] * case["d"] * (1 if case["fp8"] else 2)


def _pairs(case, lens) -> int:
    """(query token, key) pairs that attend, over the batch."""
    new = case.get("new", 0)
    if new == 0:
        return sum(lens)
    return sum(new * L + new * (new + 1) // 2 for L in lens)


def _flops(case, lens) -> float:
    return 4.0 * case["hq"] * case["d"] * _pairs(case, lens)


def _lens(case, rng: random.Random) -> list[int]:
    lo, hi = case["lo"], case["hi"]
    if case["lens"] == "uniform":
        return [rng.randint(lo, hi) for _ in range(case["batch"])]
    # Log-uniform, one sequence in ten just begun.
    out = []
    for _ in range(case["batch"]):
        if rng.random() < 0.1:
            out.append(rng.randint(1, min(15, hi)))
        else:
            out.append(_log_int(rng, max(1, lo), hi))
    return out


def _randn(shape, gen, dtype=torch.bfloat16) -> torch.Tensor:
    out = torch.empty(shape, dtype=dtype, device="cuda")
    flat = out.view(-1)
    for s in range(0, flat.numel(), GEN_CHUNK):
        n = min(GEN_CHUNK, flat.numel() - s)
        x = torch.randn(n, generator=gen, device="cuda", dtype=torch.float32)
        if dtype == torch.float8_e4m3fn:
            x.clamp_(-448.0, 448.0)
        flat[s:s + n].copy_(x.to(dtype))
    return out


def prepare(case, seed: int):
    """Pools with shuffled pages, N(0, 1) values, the batch's lengths and the call's operands."""
    rng = random.Random(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B, hq, hkv, d, P = (case[k] for k in ("batch", "hq", "hkv", "d", "page"))
    new = case.get("new", 0)
    lens = _lens(case, rng)
    width = max(1, -(-(case["hi"] + new) // P))
    pages = B * width
    table = torch.randperm(pages, generator=gen, device="cuda").to(torch.int32).view(B, width)
    dtype = torch.float8_e4m3fn if case["fp8"] else torch.bfloat16
    s = dict(case=case, lens=lens, table=table.contiguous(),
             seq_lens=torch.tensor(lens, dtype=torch.int32, device="cuda"),
             k=_randn((pages, P, hkv, d), gen, dtype), v=_randn((pages, P, hkv, d), gen, dtype))
    # Scales of an fp8 cache; a bf16 cache has none.
    s["scales"] = dict(k_scale=0.75, v_scale=1.25) if case["fp8"] else {}
    if case["kind"] == "extend":
        s["q"] = _randn((B, new, hq, d), gen)
    else:
        s["q"] = _randn((B, hq, d), gen)
    if new:
        s["k_new"] = _randn((B, new, hkv, d), gen)
        s["v_new"] = _randn((B, new, hkv, d), gen)
    if case["kind"] == "step":
        s["step"] = mx.BoundDecodeAppend(s["q"], s["k_new"], s["v_new"], s["k"], s["v"],
                                         s["table"], s["seq_lens"], **s["scales"])
    if case["kind"] == "shard":
        # The gathered partials: this GPU's (written by run) in place 0, the others' beside it.
        n = case["parts"]
        s["o_all"] = torch.randn((n, B, hq, d), generator=gen, device="cuda") * 0.05
        s["lse_all"] = torch.randn((n, B, hq), generator=gen, device="cuda") * 0.1 + \
            math.log(max(1, case["hi"])) + 0.5
    return s


def _caches(s):
    """The pools as outputs: fp8 ones as their bytes."""
    if s["case"]["fp8"]:
        return s["k"].view(torch.uint8), s["v"].view(torch.uint8)
    return s["k"], s["v"]


def run(s):
    kind = s["case"]["kind"]
    if kind == "decode":
        return mx.paged_gqa_decode(s["q"], s["k"], s["v"], s["table"], s["seq_lens"],
                                   **s["scales"])
    if kind == "step":
        return (s["step"](), *_caches(s))
    if kind == "extend":
        out = mx.paged_gqa_decode_append(s["q"], s["k_new"], s["v_new"], s["k"], s["v"],
                                         s["table"], s["seq_lens"], causal=True, **s["scales"])
        return (out, *_caches(s))
    o, lse = mx.paged_gqa_decode_partial(s["q"], s["k"], s["v"], s["table"], s["seq_lens"])
    s["o_all"][0].copy_(o)
    s["lse_all"][0].copy_(lse)
    return o, lse, mx.lse_merge(s["o_all"], s["lse_all"])


def work(case):
    # The lengths the recipe gives (their mean over a few seeds where they are random).
    seeds = range(1) if case["lo"] == case["hi"] and case["lens"] == "uniform" else range(8)
    runs = [_lens(case, random.Random(i)) for i in seeds]
    tokens = sum(sum(r) for r in runs) / len(runs)
    flops = sum(_flops(case, r) for r in runs) / len(runs)
    B, hq, hkv, d = (case[k] for k in ("batch", "hq", "hkv", "d"))
    new = case.get("new", 0)
    rows = B * hq * (new if case["kind"] == "extend" else 1)
    by = tokens * (_token_bytes(case) + 4.0 / case["page"]) + 4 * B
    by += rows * d * 2 * 2                                    # q read, out written
    by += B * new * (hkv * d * 2 * 2 + _token_bytes(case))    # new rows read, and stored
    if case["kind"] == "shard":
        by += rows * (4 * d + 4) * (1 + case["parts"])        # partial written, all parts read
    return {"bytes": by, "flops": flops}


def tolerance(case):
    # bf16 outputs (a rounding of up to 2^-9) of probabilities rounded to bf16 before the P.V
    # product: a pass over the same keys in another order differs by about 2.5e-3 relative.
    # Bytes of an fp8 pool are the nearest codes of the new rows: they stay the same.
    return {"rel": 1e-2, "max": 0.1, "differ": 0.0}


def _attend64(q, k, v, first):
    """softmax(q k^T / sqrt(d)) v in 64 bits for one KV head; query row i sees keys below
    first + i // rows_per_token.  q [T, G, d], k / v [L, d]; returns o [T, G, d], lse [T, G]."""
    T, G, d = q.shape
    L = k.shape[0]
    o = torch.empty((T, G, d), dtype=torch.float64, device=q.device)
    lse = torch.empty((T, G), dtype=torch.float64, device=q.device)
    kt = k.t().contiguous()
    step = max(1, (1 << 26) // max(1, G * L))
    pos = torch.arange(L, device=q.device)
    for t in range(0, T, step):
        n = min(step, T - t)
        s = torch.mm(q[t:t + n].reshape(n * G, d), kt) / math.sqrt(d)
        limit = (first + t + torch.arange(n, device=q.device)).repeat_interleave(G)
        s.masked_fill_(pos[None, :] >= limit[:, None], -math.inf)
        m = s.amax(1, keepdim=True)
        p = torch.exp(s - m)
        z = p.sum(1, keepdim=True)
        o[t:t + n] = (torch.mm(p, v) / z).view(n, G, d)
        lse[t:t + n] = (m + torch.log(z)).view(n, G)
    return o, lse


def exact(case, seed: int):
    s = prepare(case, seed)
    B, hq, hkv, d, P = (case[k] for k in ("batch", "hq", "hkv", "d", "page"))
    G = hq // hkv
    new = case.get("new", 0)
    T = new if case["kind"] == "extend" else 1
    q = s["q"].view(B, T, hq, d).double()
    ks, vs = s["scales"].get("k_scale", 1.0), s["scales"].get("v_scale", 1.0)
    out = torch.zeros((B, T, hq, d), dtype=torch.float64, device="cuda")
    lse = torch.full((B, T, hq), -math.inf, dtype=torch.float64, device="cuda")

    def cached(pool, b, L, scale):
        ids = s["table"][b, :-(-L // P)].long()
        return pool[ids].view(-1, hkv, d)[:L].to(torch.float64) * scale

    def appended(rows, scale):
        if not case["fp8"]:
            return rows.double()
        # Stored as the nearest e4m3fn code of x / scale (the fp32 quotient, saturated).
        x = (rows.float() / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
        return x.to(torch.float64) * scale

    for b in range(B):
        L = s["lens"][b]
        k, v = cached(s["k"], b, L, ks), cached(s["v"], b, L, vs)
        if new:
            k = torch.cat([k, appended(s["k_new"][b], ks)])
            v = torch.cat([v, appended(s["v_new"][b], vs)])
        for h in range(hkv):
            o, e = _attend64(q[b, :, h * G:(h + 1) * G], k[:, h].contiguous(),
                             v[:, h].contiguous(), L + new - T + 1)
            out[b, :, h * G:(h + 1) * G] = o
            lse[b, :, h * G:(h + 1) * G] = e
    out = out.view(s["q"].shape)
    if case["kind"] == "decode":
        return out
    if case["kind"] != "shard":
        return out, None, None
    lse = lse.view(B, hq)
    o_all, lse_all = s["o_all"].double(), s["lse_all"].double()
    o_all[0], lse_all[0] = out, lse
    w = torch.softmax(lse_all, 0)
    return out, lse, (w[..., None] * o_all).sum(0)
