"""The one-launch decode's pieces: sizes from the capacity, quarters balanced over a piece's
waves, one-piece segments, both merges, padded and packed counters -- and RoPE on K at the
positions where its two-step rotation changes base.

Against the compiled oracle under the reference checker's policy (64 BF16 ULP per element,
pyfiles/check_gqa_output.py:33-34,57-64); the path is fp64 end to end, so rows come out
within 1 ULP of the oracle's."""
from __future__ import annotations

import pytest
import torch

import attention_accelerator_amd as gqa
from attention_accelerator_amd import stimulus
from oracle import oracle as orc
from _util import assert_within_ulp, to_codes
from test_gpu_paged import _paginate

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("capacity,lengths", [
    (1024, [1, 16, 17, 64]),          # one piece: one wave, two, all four
    (1024, [65, 128, 129, 1024]),     # the last one-piece length, the first of three, sixteen
    (1040, [1040, 1025]),             # pieces of 128 keys, the last of 16 and of 1
    (2048, [2048, 1921]),             # sixteen pieces
    (4096, [2049, 4096, 4095]),       # 17 and 32 pieces: the wider merge
    (176, [176 - (i % 170) for i in range(70)]),   # 560 segments: packed counters
])
@pytest.mark.parametrize("rope_k", [False, True])
def test_pieces_match_oracle(dev, capacity, lengths, rope_k):
    b = stimulus.decode_batch(len(lengths), capacity, lengths=torch.tensor(lengths), seed=capacity + len(lengths))
    want = orc.decode(to_codes(b.q), to_codes(b.k), to_codes(b.v), b.seq_len.numpy(), b.query_pos.numpy(),
                      rope_k=rope_k)
    call = gqa.PreparedDecode(b.q.to(dev), b.k.to(dev), b.v.to(dev), b.query_pos.to(dev), b.seq_len.to(dev),
                              rope_k=rope_k)
    for _ in range(3):                # the counters return to zero
        got = to_codes(call())
        assert assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, f"cap={capacity}") <= 1


@pytest.mark.parametrize("stream", [False, True])
@pytest.mark.parametrize("length", [3, 100, 2100])
def test_rope_k_pieces_off_chunk_starts(dev, stream, length):
    """Stream-K ranges start pieces at any key, so a chunk's base position is any integer."""
    lengths = [length, max(1, length - 7), length + 5]
    b = stimulus.decode_batch(3, length + 9, lengths=torch.tensor(lengths), seed=length)
    want = orc.decode(to_codes(b.q), to_codes(b.k), to_codes(b.v), b.seq_len.numpy(), b.query_pos.numpy(),
                      rope_k=True)
    p = gqa.make_params(rope_k=True, stream_k=stream, stream_wgs=40 if stream else 0)
    got = to_codes(gqa.gqa_attention(b.q.to(dev), b.k.to(dev), b.v.to(dev), b.query_pos.to(dev), b.seq_len.to(dev),
                                     params=p))
    assert assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, f"L={length}") <= 1


# The smallest theta whose angles over 2112 positions stay within 2^26, where a chunk's rotations
# are shared; below it each pair has a sincos of its own.
_LINE = (2.0 ** 26 / 2112) ** (-128.0 / 126.0)


@pytest.mark.parametrize("path", ["single", "stream", "paged"])
@pytest.mark.parametrize("theta", [1.001 * _LINE, 0.999 * _LINE, 1e-9, 1e-12])
def test_rope_k_large_angles(dev, path, theta):
    """RoPE on K with frequencies above 1: angles about 2^26, 2^41 and 2^50 (where neighbouring
    doubles lie 1/4 rad apart), each key at its rounded angle."""
    lengths = [2100, 77, 1000]
    b = stimulus.decode_batch(3, 2112, lengths=torch.tensor(lengths), seed=17)
    want = orc.decode(to_codes(b.q), to_codes(b.k), to_codes(b.v), b.seq_len.numpy(), b.query_pos.numpy(),
                      rope_q=False, rope_k=True, theta=theta)
    p = gqa.make_params(rope_q=False, rope_k=True, theta=theta, stream_k=path == "stream")
    pos, n = b.query_pos.to(dev), b.seq_len.to(dev)
    if path == "paged":
        kp, vp, table = _paginate(b.k, b.v, b.seq_len, 17)
        got = to_codes(gqa.gqa_decode_paged(b.q.to(dev), kp.to(dev), vp.to(dev), table.to(dev), pos, n, params=p))
    else:
        got = to_codes(gqa.gqa_attention(b.q.to(dev), b.k.to(dev), b.v.to(dev), pos, n, params=p))
    assert assert_within_ulp(want.reshape(-1, 128), got.reshape(-1, 128), 64, f"{path} theta={theta}") <= 1
