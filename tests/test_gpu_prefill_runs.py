"""Key runs of the prefill attention kernel: short chunks of few sequences cut each query
block's keys into runs of whole 64-key blocks, one workgroup each, merged in fp64.

Against the compiled oracle under the reference checker's policy (64 BF16 ULP per element,
pyfiles/check_gqa_output.py:33-34,57-64), and bit for bit against a second call."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import attention_accelerator_amd as gqa
from _util import assert_within_ulp
from test_gpu_prefill import _chunk, _oracle, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,n_new,starts,q_scale", [
    (1, 17, [460], 1.0),          # 8 blocks: two runs of the shortest length
    (1, 32, [1264], 1.0),         # 21 blocks in runs of 5, the last a single block that is masked
                                  # for the first 16 queries (their running max stays -inf there)
    (1, 33, [2000], 4.0),         # a query block of one token; sharper scores
    (2, 40, [1500, 3], 1.0),      # one sequence in runs, one in a single run
    (1, 130, [511], 1.0),         # runs of cached and of chunk blocks, five query blocks
    (3, 20, [700, -1, 64], 1.0),  # an invalid start between two valid ones: NaN rows
])
def test_runs_match_oracle(dev, batch, n_new, starts, q_scale):
    cap = max(starts) + n_new + 30
    ok = [s >= 0 for s in starts]
    q, kn, vn, k, v = _chunk(batch, n_new, cap, [max(s, 0) for s in starts], 31 + n_new)
    q = (q.float() * q_scale).to(torch.bfloat16)
    st = torch.tensor(starts, dtype=torch.int32, device=dev)
    got, _, _ = _run(q, kn, vn, k, v, st, dev)
    again, _, _ = _run(q, kn, vn, k, v, st, dev)
    assert np.array_equal(got, again)
    for b in range(batch):
        if not ok[b]:
            assert (got[b] == 0x7FC0).all()
            continue
        sl = slice(b, b + 1)
        want = _oracle(q[sl], kn[sl], vn[sl], k[sl], v[sl], [starts[b]])
        assert_within_ulp(want.reshape(-1, 128), got[b].reshape(-1, 128), 64, f"T={n_new} start={starts[b]}")


def test_runs_keep_masked_keys_out(dev):
    """Chunk rows after token t, in another run's blocks or not, leave rows 0..t bit-identical."""
    starts, n_new, t = [1000], 100, 40
    q, kn, vn, k, v = _chunk(1, n_new, 1200, starts, 5)
    ref, _, _ = _run(q, kn, vn, k, v, starts, dev)
    kn2, vn2 = kn.clone(), vn.clone()
    kn2[:, t + 1:] = torch.randn(kn2[:, t + 1:].shape).to(torch.bfloat16) * 4
    vn2[:, t + 1:] = torch.randn(vn2[:, t + 1:].shape).to(torch.bfloat16) * 64
    got, _, _ = _run(q, kn2, vn2, k, v, starts, dev)
    assert np.array_equal(got[:, :t + 1], ref[:, :t + 1])


def test_runs_follow_stream_wgs(dev):
    """Four stream workgroups stand for one CU: with one CU's worth there is one run, and the
    results of both plans are within the checker's policy of each other."""
    starts, n_new = [900], 50
    q, kn, vn, k, v = _chunk(1, n_new, 1000, starts, 9)
    one = gqa.make_params(rope_k=True, stream_wgs=4)
    assert gqa.prefill_workspace_bytes(1, n_new, 1000, one) < gqa.prefill_workspace_bytes(
        1, n_new, 1000, gqa.make_params(rope_k=True, stream_wgs=1024))
    a, _, _ = _run(q, kn, vn, k, v, starts, dev, params=one)
    b, _, _ = _run(q, kn, vn, k, v, starts, dev)
    assert_within_ulp(a.reshape(-1, 128), b.reshape(-1, 128), 64, "one run against many")


def test_short_chunk_in_a_long_chunks_workspace(dev):
    """A prompt in chunks of one length and a shorter last one (cut into more runs), in the
    workspace that the long chunk asks for."""
    cap, long, short = 2100, 1024, 20
    p = gqa.make_params(rope_k=True)
    ws = torch.empty(gqa.prefill_workspace_bytes(1, long, cap, p), dtype=torch.uint8, device=dev)
    for n_new, start in ((long, 0), (short, 1500), (long, 1000)):
        q, kn, vn, k, v = _chunk(1, n_new, cap, [start], n_new + start)
        got, _, _ = _run(q, kn, vn, k, v, [start], dev, params=p, workspace=ws)
        alone, _, _ = _run(q, kn, vn, k, v, [start], dev, params=p)
        assert np.array_equal(got, alone)
        if n_new == short:
            want = _oracle(q, kn, vn, k, v, [start])
            assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, "short chunk")
