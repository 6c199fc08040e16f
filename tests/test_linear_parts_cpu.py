"""Which fp32 launches have their operands split into bf16 parts (pcb_linear_parts_form: decided on the host, nothing is launched)."""
import ctypes

import pytest
import torch

from promptcache_amd import _blocks as B

ROOM = torch.zeros(64)


def form(M, N, K, gated=False, batch=0, dtype=B.F32, off=0):
    a = B.LinearArgs(ctypes.sizeof(B.LinearArgs))
    a.dtype, a.M, a.N, a.K, a.ldx, a.ldw, a.ldy, a.epilogue = dtype, M, N, K, K, K, N, B.EPI_SILU_MUL if gated else B.EPI_STORE
    a.x = a.w = a.y = ROOM.data_ptr() + off
    a.w2 = ROOM.data_ptr() + off if gated else None
    if batch:
        a.n_batch, a.x_batch_stride, a.y_batch_stride, a.w_group_stride = batch, M * K, M * N, N * K
    return B.load().pcb_linear_parts_form(ctypes.byref(a))


# the sizes of the tests on the GPU: each tile of both epilogues is reached
@pytest.mark.parametrize("gated,M,N,K,want", [
    (False, 587, 1540, 228, 1), (False, 587, 2562, 92, 2), (False, 587, 5134, 124, 3), (True, 777, 5134, 92, 1), (True, 587, 1540, 100, 2), (True, 587, 2562, 124, 3),
    (False, 587, 1026, 1052, 1), (False, 587, 2562, 1052, 2), (False, 587, 5134, 1052, 3), (True, 587, 513, 1052, 1), (False, 587, 2562, 100, 2),
    (False, 587, 5134, 100, 3), (False, 587, 2562, 520, 2), (False, 587, 5134, 520, 3)])
def test_the_sizes_tested_reach_every_tile(gated, M, N, K, want):
    assert form(M, N, K, gated) == want


# (us, the fp32 matrix cores / in parts)
@pytest.mark.parametrize("M,N,K,gated,parts", [
    (32, 65920, 1024, False, False),    # 57.4 / 84.5: rows done for padding
    (24, 32832, 2048, False, False),    # 64.2 / 94.8
    (17, 4672, 2048, True, False),      # 29.8 / 44.4: few tiles of 32 x 16 over a deep k
    (600, 1664, 1024, False, False),    # 26.7 / 32.3: a few tiles more than the chip has CUs
    (400, 1181, 1024, True, False),     # 28.2 / 32.8
    (200, 9280, 256, False, False),     # 15.4 / 19.2
    (128, 2048, 1024, False, False),    # 64 tiles
    (600, 5136, 1024, False, True),     # 78 / 48
    (600, 2048, 1024, True, True),      # 60 / 46
    (2048, 2048, 2048, False, True),    # 147 / 96
    (100, 16448, 512, False, True)])    # 30.9 / 28.1
def test_splitting_goes_where_it_is_the_faster(M, N, K, gated, parts):
    assert bool(form(M, N, K, gated)) == parts


def test_what_cannot_be_split():
    assert form(600, 5136, 1024) and form(300, 2568, 1024, batch=4)
    assert form(600, 5136, 1024, dtype=B.BF16) == 0 and form(600, 5136, 1022) == 0 and form(600, 5136, 1024, off=8) == 0 and form(0, 5136, 1024) == 0
    assert form(600, 0, 1024) == -2001
