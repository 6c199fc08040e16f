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


def sized(M, K, N1, N2, gated):
    """The form of a pair of these sizes (results far apart)."""
    room = torch.zeros(64, dtype=torch.bfloat16)
    at, far = room.data_ptr(), 1 << 36

    def args(N, unit, y):
        a = B.LinearArgs(ctypes.sizeof(B.LinearArgs))
        a.dtype, a.M, a.N, a.K, a.ldx, a.ldw, a.ldy, a.epilogue = B.BF16, M, N, K, K, K, N, B.EPI_SILU_MUL if unit else B.EPI_STORE
        a.x = a.w = at
        a.w2, a.y, a.out_f32 = at if unit else None, y, 0 if gated else int(N == N2)
        return a
    a, b = args(N1, False, at + far), args(N2, gated, at + 2 * far)
    if gated:
        a.act_split, a.act2 = N1 // 2 // 16 * 16, B.ACT_SIGMOID
    return form(a, b)


def test_the_sizes_tested_reach_every_tile_shape():
    from tests.test_gpu_tile_pairs import SHAPES
    assert {(s[4], s[5]) for s in SHAPES} == {(False, f) for f in (2, 3, 4, 5, 6)} | {(True, f) for f in (2, 4, 6)}
    for *sizes, want in SHAPES:
        assert sized(*sizes) == want, sizes


# (us, apart / in one grid)
@pytest.mark.parametrize("M,K,N1,N2,gated,one", [
    (76, 8192, 240, 152, False, False),      # 27.3 / 43.9: a deep k over few tiles
    (323, 8192, 88, 160, False, False),      # 28.3 / 44.3
    (123, 2560, 72, 1040, False, False),     # 15.0 / 20.3
    (155, 2048, 104, 168, True, False),      # 13.6 / 18.0
    (255, 2048, 2560, 8192, False, True),    # 38.1 / 25.1
    (679, 2048, 2560, 8192, False, True),    # 52.4 / 35.0
    (558, 2048, 4096, 4096, True, True),     # 50.9 / 40.1
    (310, 512, 640, 2048, False, True)])     # 12.0 / 9.0
def test_one_grid_where_it_is_the_faster(M, K, N1, N2, gated, one):
    assert (sized(M, K, N1, N2, gated) >= TILES) == one
