"""Projections with the RMSNorm inside the launch (pc_gemm_norm.hip) against float64: one and two rows, whose operand pieces wait in LDS, and more; every number of
tiles a workgroup either kernel takes, last workgroups of fewer tiles, waves without a k-step, shares of k that no chunk of 512 divides, rows too long for LDS, pad
rows behind the live ones."""
import pytest
import torch

from tests.test_gpu_kernels import DEV, _n

pytestmark = pytest.mark.gpu
EPS = 1e-5


def inputs(M, N, K):
    g = torch.Generator().manual_seed(M * 7 + N + K)
    w = (0.05 * torch.randn(N, K, generator=g)).to(torch.float16).to(DEV)
    return w, 2.0 * torch.randn(M, K, generator=g).to(DEV), (1.0 + 0.2 * torch.randn(K, generator=g)).to(torch.float16).to(DEV)


def exact(x, gam, w):
    xd = x.double()
    return (xd * torch.rsqrt((xd * xd).mean(1, keepdim=True) + EPS) * gam.double()) @ w.double().T


# rows are split into two fp16 numbers (22 bits), products exact, sums of up to 16384 in fp32: 1e-6 of the result's size
@pytest.mark.parametrize("M", [1, 2, 3, 16])
@pytest.mark.parametrize("N,K", [(64, 32), (4096, 288), (4112, 1120), (8208, 4096), (12288, 4096), (12320, 5120), (16400, 2080), (32, 13824), (4128, 16384)])
def test_store(M, N, K):
    n = _n()
    w, x, gam = inputs(M, N, K)
    y = torch.full((M, N), 7.0, device=DEV)
    n.gemm_skinny_norm(n.to_weight_frags(w), x, gam, EPS, M, N, K, n.EPI_STORE, y=y, ldy=N)
    want = exact(x, gam, w)
    assert float((y.double() - want).norm() / want.norm()) < 1e-6
    if M > 1:                                      # rows that are not live are not read
        y2, bad = torch.full((M, N), 7.0, device=DEV), x.clone()
        bad[M - 1] = float("nan")
        n.gemm_skinny_norm(n.to_weight_frags(w), bad, gam, EPS, M, N, K, n.EPI_STORE, y=y2, ldy=N, rows_dev=torch.tensor([M - 1], dtype=torch.int32, device=DEV))
        assert torch.equal(y2[:M - 1], y[:M - 1])


@pytest.mark.parametrize("M", [1, 2, 5])
@pytest.mark.parametrize("inter,K", [(64, 96), (4096, 512), (8224, 1024), (11008, 4096), (13824, 5120), (17184, 480)])
def test_gated(M, inter, K):
    n = _n()
    w, x, gam = inputs(M, 2 * inter, K)
    hi = torch.zeros((1, inter // 32, 64, 8), dtype=torch.float16, device=DEV)
    lo = torch.zeros_like(hi)
    n.gemm_skinny_norm(n.to_weight_frags(w), x, gam, EPS, M, 2 * inter, K, n.EPI_SILU, of_hi=hi, of_lo=lo)
    z = exact(x, gam, w)
    want = torch.nn.functional.silu(z[:, :inter]) * z[:, inter:]
    got = n.from_act_frags(hi, M).double() + n.from_act_frags(lo, M).double()
    assert float((got - want).norm() / want.norm()) < 2e-6     # (and the exponential's 1e-6)


# either side of the lines between single k-steps and blocks of four: shares of two, three, four and five k-steps, nine and ten rows at two tiles a workgroup, 4096 and more of K
@pytest.mark.parametrize("M", [1, 9, 10])
@pytest.mark.parametrize("N,K", [(4800, 512), (4800, 544), (10240, 1024), (10240, 1056), (15376, 1056), (4800, 4096), (4800, 4128), (10240, 4608), (10240, 5120), (12832, 4608)])
def test_store_on_either_side_of_the_lines(M, N, K):
    test_store(M, N, K)


@pytest.mark.parametrize("M", [3, 9, 10])
@pytest.mark.parametrize("inter,K", [(4800, 1024), (4800, 1056), (11008, 4096), (11008, 4128), (11008, 4608), (13824, 4096), (13824, 4160)])
def test_gated_on_either_side_of_the_lines(M, inter, K):
    test_gated(M, inter, K)
