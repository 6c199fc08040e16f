"""Two products of the same rows in one grid of tiles (pb_linear_tiles.hip), against torch in 64 bits and the launches it stands for."""
import pytest
import torch

from promptcache_amd import _blocks as B

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rand(*shape, seed, dtype=torch.bfloat16, sd=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * sd).to(dtype).to(DEV)


# (rows, k, columns, of the second product): each tile shape, one round and more; rows, columns and k that end inside a tile, a quad, a K-step; few rows, which go out apart
SIZES = [(65, 512, 640, 2048), (129, 96, 520, 1031), (255, 1024, 1280, 4096), (300, 256, 384, 1000), (377, 2048, 2560, 8192), (640, 1024, 1030, 2052), (700, 512, 96, 3000),
         (1003, 160, 2048, 520), (1484, 256, 2560, 8192), (2195, 128, 1030, 4104), (64, 512, 640, 512)]


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("M,K,N1,N2", SIZES)
def test_pairs(gated, M, K, N1, N2):
    d = torch.float64
    x1, w1, b1, w2, b2 = rand(M, K, seed=1), rand(N1, K, seed=2, sd=K ** -0.5), rand(N1, seed=3), rand(N2, K, seed=4, sd=K ** -0.5), rand(N2, seed=5)
    x2 = x1 if gated else rand(M, K, seed=6)
    cut = N1 // 2 // 16 * 16
    want1 = x1.to(d) @ w1.to(d).T + b1.to(d)
    cache, off = torch.full((M + 3, 2 * N1), 7.0, dtype=torch.bfloat16, device=DEV), torch.tensor([2 * N1 * ((5 * m + 2) % (M + 3)) for m in range(M)],
                                                                                               dtype=torch.int64, device=DEV)
    if len(set(off.tolist())) < M:
        off = torch.arange(M, device=DEV) * (2 * N1)
    if gated:
        y1 = torch.full((M, N1), 7.0, dtype=torch.bfloat16, device=DEV)
        a = B.linear_args(x1, w1, y1, M=M, bias=b1, act_split=cut, act2=B.ACT_SIGMOID)
        want1[:, cut:] = torch.sigmoid(want1[:, cut:])
        w3, b3, y2 = rand(N2, K, seed=7, sd=K ** -0.5), rand(N2, seed=8), torch.full((M, N2), 7.0, dtype=torch.bfloat16, device=DEV)
        b = B.linear_args(x2, w2, y2, M=M, epilogue=B.EPI_SILU_MUL, w2=w3, bias=b2, bias2=b3)
        want2 = torch.nn.functional.silu(x2.to(d) @ w2.to(d).T + b2.to(d)) * (x2.to(d) @ w3.to(d).T + b3.to(d))
    else:
        y1, y2 = torch.full((M, cut), 7.0, dtype=torch.bfloat16, device=DEV), torch.full((M, N2), 7.0, device=DEV)
        a = B.linear_args(x1, w1, y1, M=M, bias=b1, split_n=cut, y2=cache, row_off2=off, head_dim2=8, head_stride2=16)
        b = B.linear_args(x2, w2, y2, M=M, bias=b2)
        want2 = x2.to(d) @ w2.to(d).T + b2.to(d)
    B.linear_pair(a, b)
    if gated:
        got1 = y1.to(d)
    else:
        c = torch.arange(N1 - cut, device=DEV)
        got1 = torch.cat([y1.to(d), cache.view(-1)[off[:, None] + (c // 8 * 16 + c % 8)[None]].to(d)], 1)
        assert int((cache != 7).sum()) <= M * (N1 - cut)             # (nothing else of the cache was written)
    # bf16 results: their rounding, 2^-9 of the value; sums of k terms of about k^-1/2 in fp32, gated: of two of them
    tol = 2e-5 if not gated else 4e-5
    assert bool(((got1 - want1).abs() <= 2 ** -8 * want1.abs() + tol).all()), float((got1 - want1).abs().max())
    step = 2 ** -8 if gated else 0.0
    assert bool(((y2.to(d) - want2).abs() <= step * want2.abs() + tol * (1 + want2.abs())).all()), float((y2.to(d) - want2).abs().max())


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_row_that_is_no_number_stays_alone(bad):
    M, K = 300, 512
    x, w1, w2 = rand(M, K, seed=1), rand(640, K, seed=2, sd=K ** -0.5), rand(2048, K, seed=3, sd=K ** -0.5)
    x[17, 5] = bad
    y1, y2 = torch.empty(M, 640, dtype=torch.bfloat16, device=DEV), torch.empty(M, 2048, device=DEV)
    B.linear_pair(B.linear_args(x, w1, y1, M=M), B.linear_args(x, w2, y2, M=M))
    rows = [r for r in range(M) if r != 17]
    assert bool(torch.isfinite(y1[rows].float()).all()) and bool(torch.isfinite(y2[rows]).all())
    assert not bool(torch.isfinite(y1[17].float()).any()) and not bool(torch.isfinite(y2[17]).any())


# what every tile shape of either epilogue takes: (rows, k, columns, of the second product, gated, pcb_linear_pair_form)
SHAPES = [(111, 96, 91, 66, False, 2), (389, 160, 3884, 4276, False, 3), (654, 160, 1945, 5955, False, 4), (786, 96, 3085, 5896, False, 5),
          (1032, 96, 3892, 5886, False, 6), (138, 352, 221, 222, True, 2), (290, 352, 3921, 5514, True, 4), (902, 352, 3501, 4123, True, 6)]


@pytest.mark.parametrize("M,K,N1,N2,gated,form", SHAPES)
def test_pairs_of_every_tile_shape(M, K, N1, N2, gated, form):
    """(That these sizes reach the shapes: test_linear_pair_cpu.py.)"""
    test_pairs(gated, M, K, N1, N2)
