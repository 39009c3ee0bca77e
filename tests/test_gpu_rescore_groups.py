"""The fp64 rescore's workgroups of four waves: keys dealt over the waves in chunks (16 keys
for a tile of four rows, 8 for a single row), items claimed past the grid, pairs past the first
64.  Against the compiled oracle under the reference checker's policy (64 BF16 ULP per
element, pyfiles/check_gqa_output.py:33-34,57-64), and bit for bit against a second call."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import attention_accelerator_amd as gqa
from _util import assert_within_ulp
from test_gpu_prefill import _chunk, _oracle, _run

pytestmark = pytest.mark.gpu


def _check(q, kn, vn, k, v, starts, dev, what, **kw):
    want = _oracle(q, kn, vn, k, v, starts)
    got, _, _ = _run(q, kn, vn, k, v, starts, dev, **kw)
    again, _, _ = _run(q, kn, vn, k, v, starts, dev, **kw)
    assert np.array_equal(got, again)
    assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, what)
    return got


@pytest.mark.parametrize("n_new,starts,wgs", [
    (1, [0, 14, 15, 16, 62, 63, 64, 130], 0),     # one tile per pair; waves and pieces with no key
    (5, [250, 3], 0),                             # tiles of a piece or a few, mixed lengths
    (3, [40] * 9, 0),                             # 72 pairs: tiles past the first 64 pairs
    (20, [70, 300], 8),                           # 320 tiles on two workgroups: claimed items
    (33, [120], 16),                              # 264 tiles on four workgroups, several pieces each
    (24, [1100, 0, 517], 0),                      # tiles short of the grid's rounds
])
def test_tiles(dev, n_new, starts, wgs):
    """Every dot product passes the fp32 range (Q scaled by 2^100, K by 2^40), so that the MFMA
    kernels' rows come out not finite and all are recomputed, four rows to a tile.  (Each row's
    weight is all on one key; spread weights below.)"""
    cap, batch = max(starts) + n_new + 5, len(starts)
    q, kn, vn, k, v = _chunk(batch, n_new, cap, starts, 11 + n_new)
    q = (q.float() * 2.0 ** 100).to(torch.bfloat16)
    kn, k = ((x.float() * 2.0 ** 40).to(torch.bfloat16) for x in (kn, k))
    p = gqa.make_params(rope_k=True, stream_wgs=wgs) if wgs else gqa.make_params(rope_k=True)
    ws = torch.empty(gqa.prefill_workspace_bytes(batch, n_new, cap, p), dtype=torch.uint8, device=dev)
    _check(q, kn, vn, k, v, starts, dev, f"tiles T={n_new}", params=p, workspace=ws)
    assert gqa.prefill_rescored_rows(ws, batch, n_new, cap, p) > 0.9 * batch * n_new * 32


@pytest.mark.parametrize("starts", [
    [0, 6, 7, 31, 63],          # up to one chunk per wave; waves with no key
    [127, 128, 500],            # pieces of 16 chunks and their remainders
    [8190],                     # a row's most pieces, merged by four waves
])
def test_rows(dev, starts):
    """One head per KV head has scores past the flag's bound: single rows (their weight on one
    key; spread weights below)."""
    q, kn, vn, k, v = _chunk(len(starts), 1, max(starts) + 8, starts, 3)
    q[:, :, ::4] = (q[:, :, ::4].float() * 2.0 ** 100).to(torch.bfloat16)
    _check(q, kn, vn, k, v, starts, dev, f"rows {starts}")


def _spread(batch, n_new, cap, starts, seed, heads, tokens):
    """N(0,1) inputs whose rows of the given heads and tokens go to the rescore with their softmax
    weights spread over all keys: K is zero in RoPE pairs 0..3 and those rows' Q is 2^20 times
    larger there, so the scores stay N(0,1) sums (a rotation keeps a pair of zeros) while the
    flag's bound on them, |q| |k| over pairs 0..7, passes 10^5."""
    q, kn, vn, k, v = _chunk(batch, n_new, cap, starts, seed)
    pairs = [0, 1, 2, 3, 64, 65, 66, 67]
    for t in (kn, k):
        t[..., pairs] = torch.where(torch.isnan(t[..., pairs]), t[..., pairs], torch.zeros(()).to(t.dtype))
    hit = torch.zeros(q.shape[1:3], dtype=torch.bool)
    hit[torch.tensor(tokens)[:, None], torch.tensor(heads)[None]] = True
    big = (q[..., pairs].float() * 2.0 ** 20).to(torch.bfloat16)
    q[..., pairs] = torch.where(hit[None, :, :, None], big, q[..., pairs])
    return (q, kn, vn, k, v), hit.numpy()


def _check_spread(dev, n_new, starts, wgs, heads, tokens):
    """The flagged rows are fp64 end to end: within 1 ULP of the oracle's, so that a wave's or a
    piece's share left out or weighted wrongly shows."""
    batch, cap = len(starts), max(starts) + n_new + 3
    args, hit = _spread(batch, n_new, cap, starts, 7 + n_new + len(starts), heads, tokens)
    p = gqa.make_params(rope_k=True, stream_wgs=wgs)
    ws = torch.empty(gqa.prefill_workspace_bytes(batch, n_new, cap, p), dtype=torch.uint8, device=dev)
    got = _check(*args, starts, dev, f"T={n_new} {starts}", params=p, workspace=ws)
    rows = gqa.prefill_rescored_rows(ws, batch, n_new, cap, p)
    # (a row of one key is that key's V: no element is small, and none is flagged)
    n_hit = sum(int(hit[max(0, 1 - st):].sum()) for st in starts)
    assert n_hit <= rows <= n_hit + max(4, 0.02 * batch * n_new * 32)
    want = _oracle(*args, starts)
    assert_within_ulp(want[:, hit].reshape(-1, 128), got[:, hit].reshape(-1, 128), 1, "flagged rows")


@pytest.mark.parametrize("n_new,starts,wgs", [
    (1, [0, 14, 15, 16, 62, 63, 64, 130], 0),     # one tile per pair; waves and pieces with no key
    (1, [5000, 2047], 0),                         # many pieces per tile, every one with weight
    (1, [3000, 700], 4096),                       # the largest grid: the most pieces
    (5, [250, 3], 0),                             # tiles of several pieces, mixed lengths
    (3, [40] * 9, 0),                             # 72 pairs: tiles past the first 64 pairs
    (20, [70, 300], 8),                           # 320 tiles on two workgroups: claimed items
    (33, [120], 16),                              # 264 tiles on four workgroups
    (24, [1100, 0, 517], 0),                      # chunk keys and cached keys in one tile
])
def test_tiles_of_spread_weights(dev, n_new, starts, wgs):
    _check_spread(dev, n_new, starts, wgs, list(range(32)), list(range(n_new)))


@pytest.mark.parametrize("n_new,starts,wgs,tokens", [
    (1, [0, 6, 7, 31, 63], 0, [0]),               # up to one chunk per wave; waves with no key
    (1, [127, 128, 500], 0, [0]),                 # pieces of 16 chunks and their remainders
    (1, [8190], 0, [0]),                          # long rows, shared by the whole grid
    (8, [3000, 40], 64, [2, 7]),                  # two rows per pair; 16 workgroups for 32 rows
    (40, [2000], 0, [0, 39]),                     # the attention kernel's rows
    (1, [300 + 37 * i for i in range(12)], 0, [0]),       # 96 rows: the same pieces for every row, a wave each
    (1, [90, 2500, 800] * 3, 4096, [0]),          # 72 rows on the largest grid: as many pieces as there are slots for
    (2, [30 + 11 * i for i in range(5)], 32, [0, 1]),     # 80 rows on eight workgroups: a piece per row, three rounds
])
def test_rows_of_spread_weights(dev, n_new, starts, wgs, tokens):
    """One head per KV head: fewer than three rows per pair, each by itself."""
    _check_spread(dev, n_new, starts, wgs, list(range(1, 32, 4)), tokens)
