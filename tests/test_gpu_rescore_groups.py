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
    kernels' rows come out not finite and all are recomputed, four rows to a tile."""
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
    """One head per KV head has scores past the flag's bound: single rows."""
    q, kn, vn, k, v = _chunk(len(starts), 1, max(starts) + 8, starts, 3)
    q[:, :, ::4] = (q[:, :, ::4].float() * 2.0 ** 100).to(torch.bfloat16)
    _check(q, kn, vn, k, v, starts, dev, f"rows {starts}")
