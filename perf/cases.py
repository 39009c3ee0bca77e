"""The work a user of this framework has it do, as measurable cases.

listed()          the named cases: smallest to largest calls of every direction the path has
draw(rng)         one more case of the same ranges
prepare(case, s)  what a program holds before the call, on the GPU, values from seed s
run(state)        one pass through the public entry points, and its outputs
exact(case, s)    the same outputs in float64 by plain torch
work(case)        the bytes and flops a pass cannot do without
tolerance(case)   how far another correct implementation at the same precision may lie

Kinds of case (field "kind"):
  golden   gqa_attention with host integers, RoPE on Q and K: the golden model's own call
  decode   PreparedDecode: one token for each sequence of a batch, post-RoPE cache
  unrotated  gqa_attention over a cache kept before RoPE (rope_k), position-major, as the
           reference core is fed: every key is rotated in the call
  paged    kv_append_paged of one token, then gqa_decode_paged: a paged serving step
  verify   PreparedPrefill of at most 16 new tokens: speculative verification
  prefill  gqa_prefill of a longer chunk over a cached prefix (or none: a fresh prompt)

A case's sizes and its sequences' lengths follow from the case alone (field "lengths" seeds
the ragged draw); a seed changes values only.
"""
import math
import random

import torch

import attention_accelerator_amd as gqa

HQ, HKV, D, BLOCK = 32, 8, 128, 16
THETA = 500000.0
ROW = HKV * D * 2 * 2          # bytes of one position's K and V rows over all KV heads
QROW = HQ * D * 2              # bytes of one token's Q (or output) rows


def listed():
    return [
        # The golden smoke case: 30 keys padded to 32 positions, the smallest real call.
        {"name": "golden_b1_len30", "kind": "golden", "batch": 1, "capacity": 32, "low": 30, "high": 30,
         "lengths": 1, "q_scale": 1.0},
        # One user's decode step at a medium context: latency.
        {"name": "decode_b1_4096", "kind": "decode", "batch": 1, "capacity": 4096, "low": 4096, "high": 4096,
         "lengths": 1, "q_scale": 1.0},
        # A serving batch with ragged contexts: the headline workload.
        {"name": "decode_b64_512_8192", "kind": "decode", "batch": 64, "capacity": 8192, "low": 512, "high": 8192,
         "lengths": 20260805, "q_scale": 1.0},
        # Long-context decode, the largest call.
        {"name": "decode_b8_131072", "kind": "decode", "batch": 8, "capacity": 131072, "low": 131072,
         "high": 131072, "lengths": 1, "q_scale": 1.0},
        # A paged serving step of a half-full server: append one token, attend.
        {"name": "paged_b24_100_6000", "kind": "paged", "batch": 24, "capacity": 6144, "low": 100, "high": 6000,
         "lengths": 3, "q_scale": 1.0},
        # A cache of unrotated keys (the reference core's contract), odd lengths, position-major.
        {"name": "unrotated_b6_77_1500", "kind": "unrotated", "batch": 6, "capacity": 1504, "low": 77, "high": 1500,
         "lengths": 5, "q_scale": 1.0},
        # One user's drafted tokens checked at once: latency.
        {"name": "verify_b1_t5_4001", "kind": "verify", "batch": 1, "new": 5, "capacity": 4096, "low": 4001,
         "high": 4001, "lengths": 1, "q_scale": 1.0},
        # Drafted tokens of a whole serving batch, short and long drafts.
        {"name": "verify_b64_t4_512_8192", "kind": "verify", "batch": 64, "new": 4, "capacity": 8192, "low": 508,
         "high": 8188, "lengths": 20260805, "q_scale": 1.0},
        {"name": "verify_b64_t16_512_8192", "kind": "verify", "batch": 64, "new": 16, "capacity": 8192, "low": 496,
         "high": 8176, "lengths": 20260805, "q_scale": 1.0},
        # Chunked prefill of four users over long contexts: the matrix-core workload.
        {"name": "prefill_b4_512_over_8192", "kind": "prefill", "batch": 4, "new": 512, "capacity": 8704,
         "low": 8192, "high": 8192, "lengths": 1, "q_scale": 1.0},
        # One user's next chunk (a follow-up message) over its conversation, odd sizes.
        {"name": "prefill_b1_200_over_5003", "kind": "prefill", "batch": 1, "new": 200, "capacity": 5248,
         "low": 5003, "high": 5003, "lengths": 1, "q_scale": 1.0},
        # Two fresh prompts with no cached prefix, sharper scores than N(0,1) gives.
        {"name": "prompt_b2_1000", "kind": "prefill", "batch": 2, "new": 1000, "capacity": 1024, "low": 0,
         "high": 0, "lengths": 1, "q_scale": 4.0},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case: kinds as in use, sizes spread over the logarithm of their range, no more
    work than the largest listed call of the kind's bound (4.3 GB of K/V, 2.8e11 flops)."""
    kind = rng.choice(["golden", "decode", "decode", "unrotated", "paged", "verify", "verify", "prefill", "prefill"])
    case = {"kind": kind, "lengths": rng.randrange(1, 1 << 30), "q_scale": rng.choice([1.0, 1.0, 4.0])}
    if kind == "golden":
        n = _log_int(rng, 1, 512)
        case.update(batch=1, capacity=(n + 15) // 16 * 16, low=n, high=n)
        return case
    if kind in ("decode", "paged"):
        batch = _log_int(rng, 1, 96)
        high = _log_int(rng, 16, min(131072, 600000 // batch))
        low = rng.choice([1, max(1, high // 8), high])
        case.update(batch=batch, low=low, high=high, capacity=(high + 31) // 16 * 16)
        return case
    if kind == "unrotated":
        batch = _log_int(rng, 1, 32)
        high = _log_int(rng, 16, min(8192, 64000 // batch))
        case.update(batch=batch, low=max(1, high // 8), high=high, capacity=(high + 31) // 16 * 16)
        return case
    if kind == "verify":
        batch, new = _log_int(rng, 1, 64), rng.randint(2, 16)
        high = _log_int(rng, 16, min(32768, 300000 // batch))
        low = rng.choice([0, high // 8, high])
        case.update(batch=batch, new=new, low=low, high=high, capacity=(high + new + 31) // 16 * 16)
        return case
    batch, new = _log_int(rng, 1, 8), _log_int(rng, 17, 1024)
    most = min(16384, 4 * 512 * 8448 // (batch * new) - new // 2)
    high = rng.choice([0, _log_int(rng, 16, max(17, most))])
    case.update(batch=batch, new=new, low=high // 4, high=high, capacity=(high + new + 31) // 16 * 16)
    return case


def _lengths(case):
    """Cached positions of each sequence (decode kinds: the cache length with the query's key)."""
    r = random.Random(case["lengths"])
    return [r.randint(case["low"], case["high"]) for _ in range(case["batch"])]


def _fresh(case):
    """Positions the call itself appends."""
    return case.get("new", 1 if case["kind"] == "paged" else 0)


def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(torch.bfloat16)


def _inputs(case, seed):
    """Q, the new K/V rows and the head-major cache [B, 8, capacity, 128] (unused rows zero, as
    an allocator leaves them), N(0,1) in BF16."""
    gen = torch.Generator("cuda").manual_seed(1000003 * int(seed) + case["lengths"] % 1000003)
    batch, cap, fresh = case["batch"], case["capacity"], _fresh(case)
    t = case.get("new")
    q = torch.randn((batch, t, HQ, D) if t else (batch, HQ, D), generator=gen, device="cuda")
    q = (q * case["q_scale"]).to(torch.bfloat16)
    k = torch.zeros((batch, HKV, cap, D), dtype=torch.bfloat16, device="cuda")
    v = torch.zeros_like(k)
    for b, n in enumerate(_lengths(case)):
        n -= fresh if case["kind"] == "paged" else 0
        if n:
            k[b, :, :n] = _randn(gen, HKV, n, D)
            v[b, :, :n] = _randn(gen, HKV, n, D)
    k_new = _randn(gen, batch, fresh, HKV, D) if fresh else None
    v_new = _randn(gen, batch, fresh, HKV, D) if fresh else None
    return q, k, v, k_new, v_new


def _blocks(case):
    """The block table of a paged case: a shuffled pool, blocks as sequences need them."""
    per = case["capacity"] // BLOCK
    ids = list(range(case["batch"] * per))
    random.Random(case["lengths"] + 1).shuffle(ids)
    return torch.tensor(ids, dtype=torch.int32).view(case["batch"], per)


def _to_pool(x, table):
    """[B, 8, capacity, 128] -> [n_blocks, 8, 16, 128] by the block table."""
    batch, _, cap, _ = x.shape
    blocks = x.view(batch, HKV, cap // BLOCK, BLOCK, D).permute(0, 2, 1, 3, 4).reshape(-1, HKV, BLOCK, D)
    pool = torch.empty_like(blocks)
    pool[table.reshape(-1).long().cuda()] = blocks
    return pool


def prepare(case, seed):
    q, k, v, k_new, v_new = _inputs(case, seed)
    kind, batch, cap = case["kind"], case["batch"], case["capacity"]
    lens = _lengths(case)
    if kind == "golden":
        return {"kind": kind, "q": q[0], "k": k[0], "v": v[0], "n": lens[0]}
    dev = torch.tensor(lens, dtype=torch.int32, device="cuda")
    if kind == "decode":
        return {"kind": kind, "call": gqa.PreparedDecode(q, k, v, dev - 1, dev)}
    if kind == "unrotated":
        k, v = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (k, v))
        return {"kind": kind, "q": q, "k": k, "v": v, "len": dev, "pos": dev - 1,
                "ws": gqa.new_workspace(batch, cap, q.device, gqa.make_params(rope_k=True))}
    if kind == "paged":
        table = _blocks(case)
        return {"kind": kind, "q": q, "k": _to_pool(k, table), "v": _to_pool(v, table), "k_new": k_new,
                "v_new": v_new, "table": table.cuda(), "len": dev, "pos": dev - 1}
    if kind == "verify":
        return {"kind": kind, "call": gqa.PreparedPrefill(q, k_new, v_new, k, v, dev), "k": k, "v": v}
    ws = torch.empty(gqa.prefill_workspace_bytes(batch, case["new"], cap), dtype=torch.uint8, device="cuda")
    return {"kind": kind, "q": q, "k": k, "v": v, "k_new": k_new, "v_new": v_new, "start": dev, "ws": ws}


def run(s):
    kind = s["kind"]
    if kind == "golden":
        return gqa.gqa_attention(s["q"], s["k"], s["v"], s["n"] - 1, s["n"], rope_q=True, rope_k=True)
    if kind == "decode":
        return s["call"]()
    if kind == "unrotated":
        return gqa.gqa_attention(s["q"], s["k"], s["v"], s["pos"], s["len"], rope_k=True, workspace=s["ws"])
    if kind == "paged":
        gqa.kv_append_paged(s["k_new"], s["v_new"], s["k"], s["v"], s["table"], s["pos"])
        out = gqa.gqa_decode_paged(s["q"], s["k"], s["v"], s["table"], s["pos"], s["len"])
        return {"out": out, "k": s["k"], "v": s["v"]}
    if kind == "verify":
        return {"out": s["call"](), "k": s["k"], "v": s["v"]}
    out = gqa.gqa_prefill(s["q"], s["k_new"], s["v_new"], s["k"], s["v"], s["start"], workspace=s["ws"])
    return {"out": out, "k": s["k"], "v": s["v"]}


def _rope(x, pos):
    """rotate_half RoPE in float64: x [..., n, 128], pos [n] float64."""
    freq = torch.tensor([THETA ** (-2.0 * i / D) for i in range(D // 2)], dtype=torch.float64, device=x.device)
    ang = pos[:, None] * freq
    c, s = ang.cos(), ang.sin()
    a, b = x[..., : D // 2], x[..., D // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def exact(case, seed):
    q, k, v, k_new, v_new = _inputs(case, seed)
    kind, t = case["kind"], case.get("new", 1)
    fresh = _fresh(case)
    out = torch.empty((case["batch"], t, HQ, D), dtype=torch.float64, device="cuda")
    k_out = k.double() if fresh else None
    v_out = v.double() if fresh else None
    for b, n in enumerate(_lengths(case)):
        start = n if kind in ("verify", "prefill") else n - 1      # position of the first query token
        total = start + t
        pos = torch.arange(start, total, dtype=torch.float64, device="cuda")
        qb = _rope(q[b].double().view(t, HKV, 4, D).permute(1, 2, 0, 3), pos) / math.sqrt(D)   # [8, 4, t, 128]
        kb, vb = k[b, :, :total].double(), v[b, :, :total].double()
        if fresh:
            kb[:, start:] = _rope(k_new[b].double().transpose(0, 1), pos)
            vb[:, start:] = v_new[b].double().transpose(0, 1)
            k_out[b, :, start:total] = kb[:, start:]
            v_out[b, :, start:total] = vb[:, start:]
        elif kind in ("golden", "unrotated"):
            kb = _rope(kb, torch.arange(total, dtype=torch.float64, device="cuda"))
        hidden = torch.arange(total, device="cuda")[None, :] > pos[:, None]
        for h in range(HKV):
            w = qb[h].reshape(4 * t, D) @ kb[h].t().contiguous()
            w = torch.softmax(w.view(4, t, total).masked_fill(hidden, -math.inf), dim=-1).view(4 * t, total)
            out[b, :, 4 * h: 4 * h + 4] = (w @ vb[h]).view(4, t, D).transpose(0, 1)
    if kind == "golden":
        return out[0, 0]
    if kind in ("decode", "unrotated"):
        return out[:, 0]
    if kind == "paged":
        table = _blocks(case)
        return {"out": out[:, 0], "k": _to_pool(k_out, table), "v": _to_pool(v_out, table)}
    return {"out": out, "k": k_out, "v": v_out}


def work(case):
    """Every K/V row a token of the sequence sees read once, Q read and the output written
    once; appended rows read once and written to the cache once.  Flops of Q.K and P.V only."""
    t, fresh = case.get("new", 1), _fresh(case)
    nbytes = case["batch"] * t * 2 * QROW
    flops = 0
    for n in _lengths(case):
        old = n - fresh if case["kind"] == "paged" else n
        nbytes += old * ROW + 2 * fresh * ROW
        if case["kind"] in ("verify", "prefill"):
            flops += 4 * D * HQ * (t * n + t * (t + 1) // 2)
        else:
            flops += 4 * D * HQ * n
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Outputs and cache rows are BF16: their own rounding is 1.7e-3 in the 2-norm (measured
    against exact()), and one unit in the last place is at most 2^-7 of a value."""
    return {"rel": 6e-3, "max": 3e-2}
