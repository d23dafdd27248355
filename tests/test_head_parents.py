"""The markov parents of the GEMM head's rows on the host side (no GPU calls: the library is a stub)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

from chain_flow_amd import _lib
from chain_flow_amd.head import ShortlistHead

V, R, D, N = 40, 256, 256, 16


class _Lib:
    """Records what the two GEMM head calls are given."""

    def __init__(self):
        self.fused = self.rows = None

    def cfh_head_packed_bytes(self, n, d, r):
        return 2 * n * (d + r)

    def cfh_head_ws_bytes(self, M, n, k):
        return 256

    def cfh_head_gemm16_markov_topk(self, x, M, d, packed, n, w1, v, prev, stride, *rest):
        ids = np.ctypeslib.as_array(C.cast(prev, C.POINTER(C.c_int32)), shape=((M - 1) * stride + 1,))[::stride]
        self.fused = ids.copy()
        return 0

    def cfh_head_gemm16_topk(self, x, M, d, packed, n, bias, k, *rest):
        if k == 0:      # the markov bias: x holds the gathered rows of w1
            self.rows = np.ctypeslib.as_array(C.cast(x, C.POINTER(C.c_uint16)), shape=(M, d)).copy()
        return 0


def _head(monkeypatch):
    stub = _Lib()
    monkeypatch.setattr(_lib, "lib", lambda: stub)
    monkeypatch.setattr(_lib, "stream_handle", lambda: None)
    h = ShortlistHead.__new__(ShortlistHead)
    h.d, h.n, h.r, h._ws = D, N, R, {}
    h.w1 = torch.arange(V, dtype=torch.float16)[:, None].expand(V, R).contiguous()
    h.w2 = torch.zeros(V, R, dtype=torch.float16)
    h.image = torch.zeros(2 * N * (D + R), dtype=torch.uint8)
    return h, stub


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64])
@pytest.mark.parametrize("M", [9, 128, 129, 256, 300])
def test_absent_markov_parents_read_the_same_row_at_every_row_count(monkeypatch, M, dtype):
    """A parent of -1 (a beam row without one) or past the table: the row count decides which launch takes
    the call, not what it reads.  The fused launch clamps int32 ids itself."""
    head, stub = _head(monkeypatch)
    prev = torch.arange(M, dtype=dtype) % V
    prev[0], prev[3], prev[M - 1] = -1, V + 2, V
    if dtype == torch.int64:
        prev[4] = 2 ** 32 + 5
    head.topk(torch.zeros(M, D, dtype=torch.float16), 4, prev=prev)
    want = prev.clamp(0, V - 1).numpy()
    if M <= 128:
        assert np.array_equal(np.clip(stub.fused, 0, V - 1), want)
    else:
        last = want[256:] if M > 256 else want
        got = stub.fused if M > 256 else stub.rows.view(np.float16)[:, 0]
        assert np.array_equal(np.clip(got, 0, V - 1), last)
        if M > 256:
            assert np.array_equal(stub.rows.view(np.float16)[:, 0], want[:256])


@pytest.mark.parametrize("M", [9, 128, 129, 256])
def test_markov_parents_on_another_device_are_refused(monkeypatch, M):
    """Parents that are not on the markov table's device never reach a launch (their address would not be
    one of the launch's device)."""
    head, stub = _head(monkeypatch)
    prev = torch.zeros(M, dtype=torch.int32, device="meta")
    with pytest.raises(RuntimeError, match="markov parents are on meta"):
        head.topk(torch.zeros(M, D, dtype=torch.float16), 4, prev=prev)
    assert stub.fused is None and stub.rows is None
