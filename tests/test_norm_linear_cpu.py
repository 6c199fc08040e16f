"""Which norms ride in the launch of the products that read them (pcb_norm_linear_takes: decided on the host, nothing is launched)."""
import ctypes

import pytest
import torch

from promptcache_amd import _blocks as B

ROOM = torch.zeros(64)
AT, FAR = ROOM.data_ptr(), 1 << 36


def takes(dtype, kind, M, K, N1, N2=0):
    """``kind``: "table", "post", "gated", or the number of streams."""
    def product(N, unit, y):
        a = B.LinearArgs(ctypes.sizeof(B.LinearArgs))
        a.dtype, a.M, a.N, a.K, a.ldx, a.ldw, a.ldy, a.epilogue = dtype, M, N, K, K, K, N, B.EPI_SILU_MUL if unit else B.EPI_STORE
        a.x, a.w, a.w2, a.y = AT, AT, AT if unit else None, y
        return a
    n = B.RowNormArgs(ctypes.sizeof(B.RowNormArgs))
    n.gain, n.gain2, n.x_out, n.eps = AT, AT, AT + 3 * FAR, 1e-6
    if kind == "table":
        n.table, n.ids, n.vocab = AT, AT, 10
    elif isinstance(kind, int):
        n.x, n.x_stride, n.coef, n.n_terms = AT, M * K, AT, kind
    else:
        n.x, n.y, n.gate, n.ldg, n.post_gain = AT, AT, AT, K, AT
    a, b = product(N1, False, AT + FAR), product(N2, kind == "gated", AT + 2 * FAR) if N2 else None
    rc = B.load().pcb_norm_linear_takes(ctypes.byref(n), ctypes.byref(a), None if b is None else ctypes.byref(b))
    assert rc in (0, B.NOT_TAKEN)
    return rc == 0


# (us, launches apart / one)
@pytest.mark.parametrize("dtype,kind,M,K,N1,N2,want", [
    (B.F32, 12, 1, 1280, 5160, 0, False),        # 11.4 / 21.2
    (B.F32, 24, 2, 64, 11976, 216, False),       # 7.3 / 12.9
    (B.F32, 7, 1, 1280, 4560, 200, False),       # 11.4 / 18.0
    (B.BF16, 24, 1, 1536, 5744, 0, False),       # 10.0 / 15.5
    (B.F32, 24, 8, 256, 96, 0, False),           # 6.5 / 9.5
    (B.BF16, 24, 3, 1024, 224, 0, False),        # 7.1 / 9.7
    (B.F32, 4, 2, 64, 11592, 0, False),          # 5.6 / 8.4
    (B.BF16, 7, 2, 768, 8064, 0, False),         # 7.8 / 8.9
    (B.BF16, 4, 1, 1024, 2560, 4096, True),      # a small model's first layers: four streams, one request
    (B.BF16, 2, 1, 1024, 2560, 8192, True),
    (B.F32, "post", 2, 1024, 5136, 0, True),
    (B.BF16, "post", 1, 2048, 5136, 0, True),
    (B.BF16, "gated", 1, 2048, 2048, 2048, True),
    (B.BF16, "gated", 8, 2048, 2048, 2048, False),
    (B.BF16, "table", 2, 1024, 5136, 0, True)])
def test_a_norm_rides_where_that_is_the_faster(dtype, kind, M, K, N1, N2, want):
    assert takes(dtype, kind, M, K, N1, N2) == want


@pytest.mark.parametrize("dtype", [B.BF16, B.F32])
def test_more_streams_ride_in_fewer_workgroups(dtype):
    for M, K in ((1, 128), (1, 512), (1, 1024), (2, 1024), (4, 512), (8, 512), (1, 2048)):
        last = None
        for terms in (1, 2, 3, 4, 5, 8, 9, 12, 13, 24):
            most = max((g for g in range(8, 1300, 8) if takes(dtype, terms, M, K, 16 * g)), default=0)
            assert last is None or most <= last
            last = most
        assert last == 0
