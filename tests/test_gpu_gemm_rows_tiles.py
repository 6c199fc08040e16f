"""Projections of 65 to 512 rows with eight, six or four weight tiles a workgroup (as many as leave no CU without one in a round): each choice at sizes around its
border, even and odd numbers of row tiles, one and two row blocks, last workgroups of fewer tiles, shares of k of no and of odd numbers of steps.  Against float64."""
import pytest
import torch

from tests.test_gpu_kernels import DEV, _n

pytestmark = pytest.mark.gpu


def operands(M, N, K):
    n, g = _n(), torch.Generator(device=DEV).manual_seed(M + N + K)
    w, x = (0.05 * torch.randn(N, K, generator=g, device=DEV)).half(), torch.randn(M, K, generator=g, device=DEV)
    hi, lo = n.to_act_frags(x)
    return n.to_weight_frags(w), hi, lo, x.double() @ w.double().T


def rel(got, want):
    return float((got.double() - want).norm() / want.norm())


# rows as two fp16 numbers (22 bits: 2^-22 / sqrt(3) in the mean), exact products, fp32 sums: 1e-6 of the result's size
@pytest.mark.parametrize("M", [65, 80, 128, 259, 288, 300, 400, 512])
@pytest.mark.parametrize("N,K,slices", [(16384, 96, 1), (16400, 160, 1), (24592, 64, 1), (12288, 224, 2), (8208, 96, 2), (4096, 160, 8), (1008, 32, 2), (16, 64, 1)])
def test_plain_stores(M, N, K, slices):
    n = _n()
    wf, hi, lo, want = operands(M, N, K)
    y = torch.full((slices, M, N), float("nan"), device=DEV)
    n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_STORE, y=y, ldy=N, kslices=slices)
    assert rel(y.sum(0), want) < 1e-6


@pytest.mark.parametrize("M", [80, 129, 288, 330])
@pytest.mark.parametrize("units,K", [(11008, 96), (8192, 160), (12304, 64), (64, 32)])
def test_feed_forwards(M, units, K):
    n = _n()
    if units % 32 == 0:
        wf, hi, lo, z = operands(M, 2 * units, K)
        oh = torch.zeros((hi.shape[0], units // 32, 64, 8), dtype=torch.float16, device=DEV)
        ol = torch.zeros_like(oh)
        n.gemm_skinny(wf, hi, lo, M, 2 * units, K, n.EPI_SILU, of_hi=oh, of_lo=ol)
        assert rel(n.from_act_frags(oh, M).double() + n.from_act_frags(ol, M).double(), torch.nn.functional.silu(z[:, :units]) * z[:, units:]) < 2e-6
        n.gemm_skinny(wf, hi, lo, M, units, K, n.EPI_GELU, of_hi=oh, of_lo=ol)
        assert rel(n.from_act_frags(oh, M).double() + n.from_act_frags(ol, M).double(), torch.nn.functional.gelu(z[:, :units])) < 2e-6
    wf, hi, lo, z = operands(M, units, K)
    y = torch.ones((M, units), device=DEV)
    n.gemm_skinny(wf, hi, lo, M, units, K, n.EPI_ADD, y=y, ldy=units)
    assert rel(y, z + 1) < 1e-6
