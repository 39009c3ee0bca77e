"""Chunked prefill (MFMA path) and KV append parity against the compiled oracle
(oracle/oracle.py prefill: the one-token golden of pyfiles/gen_gqa_wrapper_vectors.py:
121-139 per new token, new K rotated at its position and not re-rounded).

Tolerance: 64 BF16 ULP per element with the reference checker's tiny-value exemption
(pyfiles/check_gqa_output.py:33-34,57-64).  Cache rows past the chunk hold NaN, so any
read of one would poison the output."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import attention_accelerator_amd as gqa
from oracle import oracle as orc
from _util import assert_within_ulp, to_codes, to_dev, ulp_distance

pytestmark = pytest.mark.gpu


def _bf16_rne(x64: np.ndarray) -> np.ndarray:
    """double -> f32 (RNE) -> BF16 code (RNE): pyfiles/gqa_reference.py:15-19."""
    u = np.asarray(x64, dtype=np.float64).astype(np.float32).view(np.uint32).astype(np.uint64)
    return (((u + 0x7FFF + ((u >> 16) & 1)) >> 16) & 0xFFFF).astype(np.uint16)


def _chunk(batch, n_new, capacity, start, seed, device="cpu"):
    """N(0,1) BF16 inputs; cache rows < start random, rows >= start NaN."""
    g = torch.Generator("cpu").manual_seed(seed)
    q = torch.randn((batch, n_new, 32, 128), generator=g).to(torch.bfloat16)
    k_new = torch.randn((batch, n_new, 8, 128), generator=g).to(torch.bfloat16)
    v_new = torch.randn((batch, n_new, 8, 128), generator=g).to(torch.bfloat16)
    k = torch.full((batch, 8, capacity, 128), float("nan"), dtype=torch.bfloat16)
    v = torch.full((batch, 8, capacity, 128), float("nan"), dtype=torch.bfloat16)
    for b in range(batch):
        s = int(start[b])
        k[b, :, :s] = torch.randn((8, s, 128), generator=g).to(torch.bfloat16)
        v[b, :, :s] = torch.randn((8, s, 128), generator=g).to(torch.bfloat16)
    return q, k_new, v_new, k, v


def _oracle(q, k_new, v_new, k, v, start, rows=None, rope_q=True, rope_k=True):
    return orc.prefill(to_codes(q), to_codes(k), to_codes(v), to_codes(k_new), to_codes(v_new),
                       np.asarray(start), rope_q=rope_q, rope_k_new=rope_k, rows=rows)


def _run(q, k_new, v_new, k, v, start, dev, **kw):
    kd, vd = k.to(dev), v.to(dev)
    out = gqa.gqa_prefill(q.to(dev), k_new.to(dev), v_new.to(dev), kd, vd, start, **kw)
    torch.cuda.synchronize()
    return to_codes(out), kd, vd


@pytest.mark.parametrize("batch,n_new,starts,seed", [
    (2, 40, [100, 37], 1),        # ragged query block (40 = 32 + 8), chunk straddling a K block
    (1, 64, [0], 2),              # no cache: the chunk attends only to itself
    (3, 17, [5, 64, 190], 3),     # short chunk, starts at and off block boundaries
    (1, 1, [300], 4),             # one token: a decode step whose newest key is unrounded
])
def test_prefill_small_all_rows(dev, batch, n_new, starts, seed):
    cap = max(starts) + n_new + 9
    q, kn, vn, k, v = _chunk(batch, n_new, cap, starts, seed)
    want = _oracle(q, kn, vn, k, v, starts)
    got, kd, vd = _run(q, kn, vn, k, v, starts, dev)
    assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, f"prefill {batch}x{n_new}")
    # the chunk's rows landed in the cache: K rotated and rounded, V as given
    kc, vc = to_codes(kd), to_codes(vd)
    for b, s in enumerate(starts):
        for h in range(8):
            rot = orc.prepare_rows(to_codes(kn[b, :, h]), True, s)
            assert np.array_equal(kc[b, h, s:s + n_new], _bf16_rne(rot))
            assert np.array_equal(vc[b, h, s:s + n_new], to_codes(vn[b, :, h]))
        # rows past the chunk untouched (still NaN)
        assert (kc[b, :, s + n_new:] == to_codes(k[b, :, s + n_new:])).all()


@pytest.mark.parametrize("case", ["k_row_2^-10", "k_row_2^-14", "v_row_2^-14", "v_head_2^110",
                                  "k_head_2^-110", "q_head_2^100"])
def test_prefill_staging_ranges(dev, case):
    """The attention kernel reads K/V staged in fp16 with one power-of-two scale per
    64-position block.  Rows scaled far from the rest of their block, blocks whose scale
    leaves the fp32 range, and Q rows beyond it are sent to the fp64 rescore (a row 2^-10
    below its block stays on the fp16 path); every row still meets 64 ULP."""
    starts = [100, 61]
    q, kn, vn, k, v = _chunk(2, 40, 150, starts, 21)
    f = {"k_row_2^-10": 2.0 ** -10, "k_row_2^-14": 2.0 ** -14, "v_row_2^-14": 2.0 ** -14,
         "v_head_2^110": 2.0 ** 110, "k_head_2^-110": 2.0 ** -110, "q_head_2^100": 2.0 ** 100}[case]
    if case.startswith("k_row"):
        k[0, 2, 10:13] = (k[0, 2, 10:13].float() * f).to(torch.bfloat16)      # cached rows of block 0
        kn[1, 5, 3] = (kn[1, 5, 3].float() * f).to(torch.bfloat16)            # a chunk row
    elif case.startswith("v_row"):
        v[1, 6, 30:32] = (v[1, 6, 30:32].float() * f).to(torch.bfloat16)
    elif case.startswith("v_head"):
        v[0, 1, :100] = (v[0, 1, :100].float() * f).to(torch.bfloat16)
        vn[0, :, 1] = (vn[0, :, 1].float() * f).to(torch.bfloat16)
    elif case.startswith("k_head"):
        k[1, 4, :61] = (k[1, 4, :61].float() * f).to(torch.bfloat16)
        kn[1, :, 4] = (kn[1, :, 4].float() * f).to(torch.bfloat16)
    else:
        q[0, :, 9] = (q[0, :, 9].float() * f).to(torch.bfloat16)
    want = _oracle(q, kn, vn, k, v, starts)
    got, _, _ = _run(q, kn, vn, k, v, starts, dev)
    assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, f"staging {case}")


@pytest.mark.parametrize("q_scale,seed", [(16.0, 5), (64.0, 6)])
def test_prefill_peaked_scores(dev, q_scale, seed):
    """Q scaled up by a power of two (a peaked softmax: running max ~85 or ~340 in log2
    units against ~6 for N(0,1)).  The kernel's scores are fp32 sums whose error grows with
    the scores, so the rows it sends to the fp64 rescore must follow the row's max: every
    element within 64 ULP of the oracle, all 200 tokens of both sequences."""
    starts = [1500, 2300]
    q, k_new, v_new, k, v = _chunk(2, 100, 2500, starts, seed)
    q = (q.float() * q_scale).to(torch.bfloat16)
    want = _oracle(q, k_new, v_new, k, v, starts, rope_q=False)
    got, _, _ = _run(q, k_new, v_new, k, v, starts, dev, rope_q=False)
    assert_within_ulp(want, got, 64, f"prefill, Q x{q_scale:g}")


def test_prefill_no_rope(dev):
    starts = [70, 150]
    q, kn, vn, k, v = _chunk(2, 33, 200, starts, 5)
    want = _oracle(q, kn, vn, k, v, starts, rope_q=False, rope_k=False)
    got, kd, _ = _run(q, kn, vn, k, v, starts, dev, rope_q=False, rope_k=False)
    assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, "prefill no rope")
    assert np.array_equal(to_codes(kd)[0, 3, 70:103], to_codes(kn[0, :, 3]))


def test_prefill_many_sequences(dev):
    """70 sequences of 20 new tokens after 0..300 cached positions (560 (sequence, KV head)
    pairs: staging, the block-statistics reduction and the attention grid over more than 64
    sequences): every output row against the oracle."""
    g = torch.Generator("cpu").manual_seed(61)
    starts = [int(x) for x in torch.randint(0, 301, (70,), generator=g)]
    q, kn, vn, k, v = _chunk(70, 20, max(starts) + 20, starts, 61)
    want = _oracle(q, kn, vn, k, v, starts)
    got, _, _ = _run(q, kn, vn, k, v, starts, dev)
    assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, "prefill B=70 T=20")


def test_multi_token_decode_ragged_batch(dev):
    """Multi-token decode (T=4 new tokens per sequence, e.g. speculative drafts) over a
    ragged batch of 8 sequences with 100..3000 cached positions, through gqa_prefill:
    every output row against the oracle's per-token reference step."""
    g = torch.Generator("cpu").manual_seed(13)
    starts = [int(x) for x in torch.randint(100, 3001, (8,), generator=g)]
    q, kn, vn, k, v = _chunk(8, 4, 3004, starts, 13)
    want = _oracle(q, kn, vn, k, v, starts)
    got, _, _ = _run(q, kn, vn, k, v, starts, dev)
    w = assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, "multi-token decode")
    print("worst ULP", w)


def test_prefill_position_major_cache(dev):
    """Cache stored [B][S][8][128] (position-major): same bits as head-major, and the chunk's
    rows land at the right (position, head)."""
    starts = [45, 130]
    q, kn, vn, k, v = _chunk(2, 24, 180, starts, 12)
    want, kd_ref, _ = _run(q, kn, vn, k, v, starts, dev)
    kp = k.permute(0, 2, 1, 3).contiguous().to(dev).permute(0, 2, 1, 3)
    vp = v.permute(0, 2, 1, 3).contiguous().to(dev).permute(0, 2, 1, 3)
    got = to_codes(gqa.gqa_prefill(q.to(dev), kn.to(dev), vn.to(dev), kp, vp, starts))
    torch.cuda.synchronize()
    assert np.array_equal(got, want)
    assert np.array_equal(to_codes(kp), to_codes(kd_ref))


def test_prefill_causal_independence(dev):
    """Token t's output does not depend on chunk rows after t (masked keys contribute
    exactly zero): perturbing rows t+1.. leaves rows 0..t bit-identical."""
    starts = [200]
    q, kn, vn, k, v = _chunk(1, 96, 300, starts, 6)
    ref, _, _ = _run(q, kn, vn, k, v, starts, dev)
    t = 45
    kn2, vn2, q2 = kn.clone(), vn.clone(), q.clone()
    kn2[:, t + 1:] = torch.randn(kn2[:, t + 1:].shape).to(torch.bfloat16) * 4
    vn2[:, t + 1:] = torch.randn(vn2[:, t + 1:].shape).to(torch.bfloat16) * 4
    q2[:, t + 1:] = 0
    got, _, _ = _run(q2, kn2, vn2, k, v, starts, dev)
    assert np.array_equal(got[:, :t + 1], ref[:, :t + 1])


def test_prefill_deterministic_and_workspace_reuse(dev):
    starts = [128, 0, 77]
    q, kn, vn, k, v = _chunk(3, 50, 180, starts, 7)
    a, _, _ = _run(q, kn, vn, k, v, starts, dev)
    ws = torch.empty(gqa.prefill_workspace_bytes(3, 50, k.shape[2]), dtype=torch.uint8, device=dev)
    ws.fill_(0xFF)
    b, _, _ = _run(q, kn, vn, k, v, starts, dev, workspace=ws)
    assert np.array_equal(a, b)


def test_prepared_prefill_matches_and_repeats(dev):
    """PreparedPrefill (arguments bound once) gives the bits of gqa_prefill, call after call
    on the same cache (each call rewrites the chunk's rows with the same values)."""
    starts = [96, 3]
    q, kn, vn, k, v = _chunk(2, 40, 160, starts, 11)
    want, _, _ = _run(q, kn, vn, k, v, starts, dev)
    kd, vd = k.to(dev), v.to(dev)
    call = gqa.PreparedPrefill(q.to(dev), kn.to(dev), vn.to(dev), kd, vd,
                               torch.tensor(starts, dtype=torch.int32, device=dev))
    for _ in range(3):
        got = to_codes(call())
        torch.cuda.synchronize()
        assert np.array_equal(got, want)


def test_prefill_invalid_device_start_gives_nan_rows(dev):
    starts = torch.tensor([40, 500], dtype=torch.int32)     # sequence 1: 500 + 20 > capacity
    q, kn, vn, k, v = _chunk(2, 20, 100, [40, 0], 8)
    kd, vd = k.to(dev), v.to(dev)
    out = gqa.gqa_prefill(q.to(dev), kn.to(dev), vn.to(dev), kd, vd, starts.to(dev))
    torch.cuda.synchronize()
    got = to_codes(out)
    assert (got[1] == 0x7FC0).all()
    assert np.array_equal(to_codes(kd)[1], to_codes(k)[1])   # cache of sequence 1 untouched
    want = _oracle(q[:1], kn[:1], vn[:1], k[:1], v[:1], [40])
    assert_within_ulp(want.reshape(-1, 128), got[:1].reshape(-1, 128), 64, "valid next to invalid")


def test_prefill_host_validation_rejects(dev):
    q, kn, vn, k, v = _chunk(1, 10, 50, [0], 9)
    kd, vd = k.to(dev), v.to(dev)
    for st in ([-1], [41]):
        with pytest.raises(gqa.GqaConfigError):
            gqa.gqa_prefill(q.to(dev), kn.to(dev), vn.to(dev), kd, vd, st)


def test_prefill_config5_sampled_rows(dev):
    """B=4, 512 new tokens after an 8192-token post-RoPE cache (8704 keys for the last
    token): 64 rows of every sequence against the oracle -- in each of the 16 query blocks
    of 32 tokens its first and last row and two more drawn per sequence (511 included) --
    every output finite, a second call bit-identical."""
    starts = [8192] * 4
    g = torch.Generator("cuda").manual_seed(20260805)
    shape_q, shape_n = (4, 512, 32, 128), (4, 512, 8, 128)
    q = torch.randn(shape_q, generator=g, device=dev).to(torch.bfloat16)
    kn = torch.randn(shape_n, generator=g, device=dev).to(torch.bfloat16)
    vn = torch.randn(shape_n, generator=g, device=dev).to(torch.bfloat16)
    k = torch.full((4, 8, 8704, 128), float("nan"), dtype=torch.bfloat16, device=dev)
    v = torch.full_like(k, float("nan"))
    k[:, :, :8192] = torch.randn((4, 8, 8192, 128), generator=g, device=dev).to(torch.bfloat16)
    v[:, :, :8192] = torch.randn((4, 8, 8192, 128), generator=g, device=dev).to(torch.bfloat16)
    k_host, v_host = k.cpu(), v.cpu()
    out = gqa.gqa_prefill(q, kn, vn, k, v, starts)
    out2 = gqa.gqa_prefill(q, kn, vn, k, v, starts)
    got = to_codes(out)
    assert np.array_equal(got, to_codes(out2))
    assert np.isfinite(out.float().cpu().numpy()).all()
    rng = np.random.default_rng(5)
    qc, kc, vc, knc, vnc = (to_codes(t) for t in (q, k_host, v_host, kn, vn))
    worst_ulp, worst_abs = 0, 0.0
    for b in range(4):
        rows = sorted({r for j in range(16)
                       for r in (32 * j, 32 * j + 31, *(32 * j + rng.choice(np.arange(1, 31), 2, replace=False)))})
        assert len(rows) == 64 and rows[-1] == 511
        want, want64 = orc.prefill(qc[b:b + 1], kc[b:b + 1], vc[b:b + 1], knc[b:b + 1], vnc[b:b + 1],
                                   np.asarray(starts[b:b + 1]), rows=rows, want_f64=True)
        gr = got[b:b + 1, rows]
        w = assert_within_ulp(want.reshape(-1, 128), gr.reshape(-1, 128), 64, f"config 5 sequence {b}")
        gv = (gr.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
        worst_ulp, worst_abs = max(worst_ulp, w), max(worst_abs, float(np.abs(gv - want64).max()))
    print(f"config 5: worst {worst_ulp} ULP, max |err| vs float64 golden {worst_abs:.3e}")


def test_kv_append_then_decode(dev):
    """Append one token per sequence with RoPE on insert, then decode over the grown
    cache: equals the oracle on the cache the append wrote (a post-RoPE cache)."""
    starts = [31, 500, 257]
    cap = 520
    q, kn, vn, k, v = _chunk(3, 1, cap, starts, 10)
    kd, vd = k.to(dev), v.to(dev)
    gqa.kv_append(kn.to(dev), vn.to(dev), kd, vd, starts)
    torch.cuda.synchronize()
    kc, vc = to_codes(kd), to_codes(vd)
    for b, s in enumerate(starts):
        for h in range(8):
            rot = orc.prepare_rows(to_codes(kn[b, :, h]), True, s)
            assert np.array_equal(kc[b, h, s:s + 1], _bf16_rne(rot))
            assert np.array_equal(vc[b, h, s:s + 1], to_codes(vn[b, :, h]))
    seq_len = [s + 1 for s in starts]
    qd = q[:, 0].to(dev)
    got = to_codes(gqa.gqa_attention(qd, kd, vd, starts, seq_len))
    want = orc.decode(to_codes(q[:, 0]), kc, vc, np.asarray(seq_len), np.asarray(starts))
    assert_within_ulp(want, got, 64, "append then decode")


def test_prefill_chunk_blocks_meet_in_fp64(dev):
    """Chunk keys 64..127 repeat keys 0..63 with V negated, the later keys have weights of about
    2^-16: a row from token 192 on is the later keys' share alone, about 3 * 10^-6 of what the
    first two blocks add and take back.  Where the blocks meet in fp64, one's fp32 sum is the
    other's negative, but for a last bit in a few elements of a hundred; where one is summed onto
    the other in fp32, most elements are left with an error of that bit, 2^-24 / 3 * 10^-6 = 2 %
    of them or several ULP (53 in 100 measured; 3 with fp64).  Few of these rows go to the
    rescore: no element is far below its row."""
    n_new = 224
    q, kn, vn, k, v = _chunk(1, n_new, n_new + 5, [0], 41)
    q[:] = q[:, :1, ::4].repeat_interleave(4, dim=2)              # one query vector per KV head
    kn[:, 64:128] = kn[:, :64]
    kn[:, 128:] = -q[:, :1, ::4]
    vn[:, 64:128] = -vn[:, :64]
    ws = torch.empty(gqa.prefill_workspace_bytes(1, n_new, n_new + 5), dtype=torch.uint8, device=dev)
    want = _oracle(q, kn, vn, k, v, [0], rope_q=False, rope_k=False)
    got, _, _ = _run(q, kn, vn, k, v, [0], dev, rope_q=False, rope_k=False, workspace=ws)
    rows = gqa.prefill_rescored_rows(ws, 1, n_new, n_new + 5)
    print(f"{rows} of {n_new * 32} rows rescored", flush=True)
    off = ulp_distance(want[:, 192:], got[:, 192:]) > 1
    assert off.mean() < 0.15, f"{int(off.sum())} of {off.size} elements more than 1 ULP off"
    assert rows < 100


def test_prefill_two_byte_aligned_inputs(dev):
    """Q and the new K/V rows at 2-byte (not 16-byte) aligned addresses: the same bits as aligned
    inputs, in rows that the attention kernel ends and in rows of the rescore (a Q head 2^100
    times larger)."""
    starts = [300, 9]
    q, kn, vn, k, v = _chunk(2, 40, 345, starts, 48)
    q[:, :, 6] = (q[:, :, 6].float() * 2.0 ** 100).to(torch.bfloat16)
    want, _, _ = _run(q, kn, vn, k, v, starts, dev)

    def shifted(x):
        flat = torch.empty(x.numel() + 1, dtype=x.dtype, device=dev)
        view = flat[1:].view(x.shape)
        view.copy_(x.to(dev))
        return view

    qs, kns, vns = shifted(q), shifted(kn), shifted(vn)
    assert qs.data_ptr() % 16 != 0 and kns.data_ptr() % 16 != 0
    got = to_codes(gqa.gqa_prefill(qs, kns, vns, k.to(dev), v.to(dev), starts))
    torch.cuda.synchronize()
    assert np.array_equal(got, want)
