"""Decode with host lengths (gqa_decode_host_bf16, and gqa_attention with Python integers):
the same bits as the call with device lengths, whatever the workspace holds; bad lengths are
rejected before anything is launched."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import attention_accelerator_amd as gqa
from attention_accelerator_amd import _lib, stimulus
from attention_accelerator_amd._lib import GqaKvLayout
from _util import to_codes


@pytest.mark.gpu
@pytest.mark.parametrize("batch,capacity,low", [
    (1, 32, 30),          # lengths with the launch, one piece, no counter
    (8, 160, 1),          # the most sequences that travel so; counted segments among them
    (9, 160, 1),          # one more: lengths stored by a launch of their own
    (3, 20000, 500),      # the three-launch plan
    (1001, 16, 1),        # lengths of more than one launch, packed counters
])
def test_host_lengths_match_device_lengths(dev, batch, capacity, low):
    b = stimulus.decode_batch(batch, capacity, min_len=low, max_len=capacity, seed=batch)
    q, k, v = b.q.to(dev), b.k.to(dev), b.v.to(dev)
    pos = torch.clamp(b.query_pos - torch.arange(batch, dtype=torch.int32) % 3, min=0)   # causal below padding too
    want = gqa.gqa_attention(q, k, v, pos.to(dev), b.seq_len.to(dev), rope_k=True)
    got = gqa.gqa_attention(q, k, v, pos.tolist(), b.seq_len.tolist(), rope_k=True)
    assert np.array_equal(to_codes(got), to_codes(want))
    p = gqa.make_params(rope_k=True)
    L = _lib.lib()
    nbytes = L.gqa_decode_host_workspace_bytes(ctypes.byref(p), batch, capacity)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=dev)
    lay = GqaKvLayout(k.stride(0), k.stride(1), k.stride(2), capacity)
    sl, qp = b.seq_len.contiguous(), pos.contiguous()
    for _ in range(2):
        out = torch.zeros_like(want)
        st = L.gqa_decode_host_bf16(ctypes.byref(p), q.data_ptr(), k.data_ptr(), v.data_ptr(), ctypes.byref(lay),
                                    sl.data_ptr(), qp.data_ptr(), batch, out.data_ptr(), ws.data_ptr(), nbytes,
                                    torch.cuda.current_stream().cuda_stream)
        assert st == 0
        assert np.array_equal(to_codes(out), to_codes(want))


@pytest.mark.parametrize("seq_len,query_pos,status", [
    ([0], [0], 1), ([33], [0], 1), ([5], [5], 1), ([5], [-1], 1),     # gqa_validate_lengths
    ([5], [4], 3),                                                     # workspace too small
])
def test_host_lengths_rejected_before_launch(seq_len, query_pos, status):
    p = gqa.make_params()
    L = _lib.lib()
    lay = GqaKvLayout(8 * 32 * 128, 32 * 128, 128, 32)
    buf = (ctypes.c_char * 4096)()
    base = (ctypes.addressof(buf) + 255) // 256 * 256      # aligned; never read: nothing is launched
    sl, qp = (ctypes.c_int32 * 1)(*seq_len), (ctypes.c_int32 * 1)(*query_pos)
    st = L.gqa_decode_host_bf16(ctypes.byref(p), base, base, base, ctypes.byref(lay), ctypes.addressof(sl),
                                ctypes.addressof(qp), 1, base, base, 256, None)
    assert st == status
