"""How two products of the same rows go out (pcb_linear_pair_form: decided on the host, nothing is launched): results that overlap what the other product
reads or stores go in two launches, one after the other."""
import ctypes

import pytest
import torch

from promptcache_amd import _blocks as B

TWO, FEW, TILES = 0, 1, 2


@pytest.fixture(autouse=True)
def host_tensors(monkeypatch):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)               # (only addresses are looked at)


def form(a, b):
    return B.load().pcb_linear_pair_form(ctypes.byref(a), ctypes.byref(b))


def bf(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


@pytest.mark.parametrize("M,together", [(4, FEW), (377, TILES)])
def test_products_that_meet_in_memory_go_one_after_the_other(M, together):
    K, N1, N2 = 512, 640, 2048
    x1, x2, w1, w2, y1, y2 = bf(M, K), bf(M, K), bf(N1, K), bf(N2, K), bf(M, N1), bf(M, N2)
    P = lambda x, w, y, **kw: B.linear_args(x, w, y, M=M, **kw)     # noqa: E731
    a, b = P(x1, w1, y1), P(x2, w2, y2)
    assert (form(a, b) if together == FEW else min(form(a, b), TILES)) == together
    assert form(P(x1, w1, y1), P(x1, w2, y2)) == form(a, b)          # (the same rows)
    flat = bf(4 * M * N2)
    rows = lambda at, cols: flat[at:at + M * cols].view(M, cols)    # noqa: E731
    # the second's input is the first's result, or a part of it; the first's input is the second's result
    assert form(P(x1, w1, rows(0, N1)), P(rows(8, K), w2, y2)) == TWO
    assert form(P(rows(M * N2 - 8, K), w1, y1), P(x2, w2, rows(0, N2))) == TWO
    assert form(P(rows(M * N2, K), w1, y1), P(x2, w2, rows(0, N2))) == form(a, b)
    # results that meet, by one piece of 16 bytes and by none; fp32 results are twice as long
    assert form(P(x1, w1, rows(0, N1)), P(x2, w2, rows(M * N1 - 8, N2))) == TWO
    assert form(P(x1, w1, rows(0, N1)), P(x2, w2, rows(M * N1, N2))) == form(a, b)
    wide = flat.view(torch.float32)[:M * N2].view(M, N2)
    assert form(P(x1, w1, rows(2 * M * N2 - 8, N1)), P(x2, w2, wide)) == TWO
    assert form(P(x1, w1, rows(2 * M * N2, N1)), P(x2, w2, wide)) >= FEW
    # split-off columns as fp32 rows
    tail = flat.view(torch.float32)[:M * 128].view(M, 128)
    cut = dict(split_n=N1 - 128, y2=tail, head_stride2=128, y2_f32=True)
    assert form(P(x1, w1, bf(M, N1 - 128), **cut), P(rows(2 * M * 128 - 8, K), w2, y2)) == TWO
    assert form(P(x1, w1, bf(M, N1 - 128), **cut), P(x2, w2, rows(2 * M * 128 - 8, N2))) == TWO
    assert form(P(x1, w1, bf(M, N1 - 128), **cut), P(rows(2 * M * 128, K), w2, y2)) >= FEW
    # the gated unit's gate per row
    if M == 377:
        gated = dict(epilogue=B.EPI_SILU_MUL, w2=bf(N2, K))
        apart = form(a, P(x2, w2, y2, row_gate=bf(M, 1), **gated))
        assert apart >= TILES
        assert form(P(x1, w1, rows(0, N1)), P(x2, w2, y2, row_gate=rows(0, N1)[:, 5:6], ld_row_gate=N1, **gated)) == TWO
