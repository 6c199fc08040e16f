"""Projections of up to 32 rows with the next k-steps under way (pc_gemm_pipe.hip), and where five tiles or two pairs a workgroup are taken, against float64: both
numbers of row tiles, last workgroups of fewer tiles, shares of k of no, one, two and many steps, slices, every epilogue but the rotation's (its bits are those of
the launches apart: test_gpu_kernels.py), pad rows behind the live ones."""
import pytest
import torch

from tests.test_gpu_kernels import DEV, _n

pytestmark = pytest.mark.gpu


def operands(M, N, K):
    n, g = _n(), torch.Generator().manual_seed(M + N + K)
    w, x = (0.05 * torch.randn(N, K, generator=g)).to(torch.float16).to(DEV), torch.randn(M, K, generator=g).to(DEV)
    mt = 4 if M > 32 else (M + 15) // 16
    hi = torch.zeros((mt, K // 32, 64, 8), dtype=torch.float16, device=DEV)
    lo = torch.zeros_like(hi)
    n.rmsnorm_frag(x.clone(), torch.ones(K, dtype=torch.float16, device=DEV), hi, lo, M, K, 0.0)     # (rows of mean square 1, as two fp16 planes)
    xd = x.double()
    return n.to_weight_frags(w), hi, lo, (xd * torch.rsqrt((xd * xd).mean(1, keepdim=True))) @ w.double().T


def rel(got, want):
    return float((got.double() - want).norm() / want.norm())


# rows as two fp16 numbers (22 bits), exact products, fp32 sums of up to 16384: 1e-6 of the result's size; 65 .. 80 tiles of 16 take one to five a workgroup by what
# the chip has places for, so the sizes say which: 768 three, 784 and 960 four, 1024 over K = 2048 five, 320 in four slices five
@pytest.mark.parametrize("M", [1, 13, 17, 32, 33, 64])
@pytest.mark.parametrize("N,K,slices", [(12288, 96, 1), (12240, 288, 1), (12544, 2560, 1), (15376, 1120, 1), (16384, 2048, 1), (14000, 4096, 1), (5120, 2080, 4), (4096, 1376, 4), (5008, 160, 4)])
def test_stores_and_sums(M, N, K, slices):
    n = _n()
    wf, hi, lo, want = operands(M, N, K)
    y = torch.zeros((slices, M, N), device=DEV)
    n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_STORE, y=y, ldy=N, kslices=slices)
    assert rel(y.sum(0), want) < 1e-6
    if slices == 1:
        z = torch.ones((M, N), device=DEV)
        n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_ADD, y=z, ldy=N)
        assert rel(z, want + 1) < 1e-6
        if N % 32 == 0:
            mt = hi.shape[0]
            oh = torch.zeros((mt, N // 32, 64, 8), dtype=torch.float16, device=DEV)
            ol = torch.zeros_like(oh)
            n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_GELU, of_hi=oh, of_lo=ol)
            assert rel(n.from_act_frags(oh, M).double() + n.from_act_frags(ol, M).double(), torch.nn.functional.gelu(want)) < 2e-6
        if 1 < M <= 32:                            # rows that are not live are not read
            y2 = torch.zeros((M, N), device=DEV)
            bad = hi.clone()
            bad[(M - 1) // 16, :, [16 * g + (M - 1) % 16 for g in range(4)]] = float("nan")
            n.gemm_skinny(wf, bad, lo, M, N, K, n.EPI_STORE, y=y2, ldy=N, rows_dev=torch.tensor([M - 1], dtype=torch.int32, device=DEV))
            assert torch.equal(y2[:M - 1], y[0, :M - 1])


@pytest.mark.parametrize("M", [12, 20, 40, 64])
@pytest.mark.parametrize("inter,K", [(11008, 512), (13824, 1056), (12320, 96), (64, 32)])
def test_gated(M, inter, K):
    n = _n()
    wf, hi, lo, z = operands(M, 2 * inter, K)
    oh = torch.zeros((hi.shape[0], inter // 32, 64, 8), dtype=torch.float16, device=DEV)
    ol = torch.zeros_like(oh)
    n.gemm_skinny(wf, hi, lo, M, 2 * inter, K, n.EPI_SILU, of_hi=oh, of_lo=ol)
    want = torch.nn.functional.silu(z[:, :inter]) * z[:, inter:]
    assert rel(n.from_act_frags(oh, M).double() + n.from_act_frags(ol, M).double(), want) < 2e-6


# K slices added inside the launch, four and eight tiles a workgroup: the next k-step under way
@pytest.mark.parametrize("M", [1, 12, 16])
@pytest.mark.parametrize("N,K,S,T", [(5120, 13824, 3, 4), (5120, 5120, 3, 4), (6656, 1024, 2, 4), (6672, 288, 3, 8), (80, 32, 3, 4)])
def test_slices_added_in_the_launch(M, N, K, S, T):
    n = _n()
    wf, hi, lo, want = operands(M, N, K)
    y = torch.ones((M, N), device=DEV)
    scratch = torch.empty(n.gemm_skinny_ks_scratch_bytes(N, 8) // 4, device=DEV)
    counters = torch.zeros(N // 16, dtype=torch.int32, device=DEV)
    for k in range(1, 4):
        n.gemm_skinny_ks(wf, hi, lo, M, N, K, y, N, S, T, scratch, counters)
        assert rel(y, 1 + k * want) < 2e-6 and not bool(counters.any())


# 33 to 64 rows, a vocabulary of a short k (four tiles a workgroup), the last workgroup with fewer; one plane too
@pytest.mark.parametrize("M", [33, 47, 64])
@pytest.mark.parametrize("N,K", [(32000, 96), (32016, 288), (24592, 32)])
def test_vocabularies(M, N, K):
    n = _n()
    wf, hi, lo, want = operands(M, N, K)
    y = torch.zeros((M, N), device=DEV)
    n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_STORE, y=y, ldy=N)
    assert rel(y, want) < 1e-6
    n.gemm_skinny(wf, hi, None, M, N, K, n.EPI_STORE, y=y, ldy=N)          # (rows rounded to 11 bits: a uniform error of 2^-12 at most, 2^-12 / sqrt(3) in the mean)
    assert rel(y, want) < 2.0 ** -12


# either side of the lines between the next k-steps under way and blocks one after the other: shares of an odd and an even number of blocks, 4096 and more of K, gated ones
@pytest.mark.parametrize("M", [12, 16, 17, 32])
@pytest.mark.parametrize("N,K,slices", [(8992, 768, 1), (12832, 1536, 1), (12832, 4096, 1), (12832, 4128, 1), (8992, 4608, 1), (8992, 5120, 1), (4096, 2560, 4)])
def test_stores_on_either_side_of_the_lines(M, N, K, slices):
    test_stores_and_sums(M, N, K, slices)


@pytest.mark.parametrize("M,N,K", [(24, 8336, 3072), (25, 8336, 3072), (32, 12288, 3072), (25, 12544, 3072)])
def test_more_than_24_rows_over_an_odd_multiple_of_1024(M, N, K):
    test_stores_and_sums(M, N, K, 1)


@pytest.mark.parametrize("M", [16, 17])
@pytest.mark.parametrize("inter,K", [(11008, 1024), (11008, 1056), (11008, 4096), (13824, 4096), (13824, 4128)])
def test_gated_on_either_side_of_the_lines(M, inter, K):
    test_gated(M, inter, K)


# eight tiles a workgroup from K = 1536 on, in slices only while they are one round of the chip
@pytest.mark.parametrize("M", [33, 47, 64])
@pytest.mark.parametrize("N,K,slices", [(32016, 1504, 1), (32016, 1536, 1), (24592, 1568, 1), (9232, 3072, 2), (9232, 3008, 2), (15360, 4608, 3)])
def test_vocabularies_on_either_side_of_the_lines(M, N, K, slices):
    test_stores_and_sums(M, N, K, slices)
