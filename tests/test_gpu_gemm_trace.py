"""pc_dev_gemm_trace: every weight-streaming launch of up to 64 rows stamps its workgroups' times, whichever kernel it is, and leaves its results as they are."""
import pytest
import torch

from tests.test_gpu_gemm_norm import EPS, inputs
from tests.test_gpu_gemm_pipe import operands
from tests.test_gpu_kernels import DEV, _n

pytestmark = pytest.mark.gpu


def stamped(run, room=4096):
    """Stamps [workgroups that have any][8 waves][entry, products done, reduced, stored] of one launch."""
    n = _n()
    buf = torch.zeros(room * 32, dtype=torch.int64, device=DEV)
    n.load().pc_dev_gemm_trace(buf.data_ptr())
    try:
        run()
    finally:
        n.load().pc_dev_gemm_trace(None)
    t = buf.view(room, 8, 4).cpu()
    return t[(t > 0).any(-1).any(-1)]


def look(t, workgroups):
    assert t.shape[0] == workgroups
    assert bool((t[:, :, :3] > 0).all()) and bool((t[:, :, 1] >= t[:, :, 0]).all()) and bool((t[:, :, 2] >= t[:, :, 1]).all())
    stored = t[:, :, 3] > 0
    assert bool(stored[:, 0].all()) and bool((t[:, :, 3] >= t[:, :, 2])[stored].all())


@pytest.mark.parametrize("M,workgroups", [(1, 256), (2, 256), (3, 256), (16, 256)])
def test_normed(M, workgroups):
    n, (N, K) = _n(), (12288, 1120)                                  # 768 tiles: three a workgroup
    w, x, gam = inputs(M, N, K)
    wf, y, z = n.to_weight_frags(w), torch.zeros((M, N), device=DEV), torch.zeros((M, N), device=DEV)
    n.gemm_skinny_norm(wf, x, gam, EPS, M, N, K, n.EPI_STORE, y=z, ldy=N)
    look(stamped(lambda: n.gemm_skinny_norm(wf, x, gam, EPS, M, N, K, n.EPI_STORE, y=y, ldy=N)), workgroups)
    assert torch.equal(y, z)


@pytest.mark.parametrize("M", [5, 20, 40])
@pytest.mark.parametrize("N,K,slices,workgroups", [(12288, 1120, 1, 256), (5120, 2080, 4, 256), (1024, 288, 1, 64)])
def test_two_planes(M, N, K, slices, workgroups):
    n = _n()
    wf, hi, lo, _ = operands(M, N, K)
    y, z = torch.zeros((slices, M, N), device=DEV), torch.zeros((slices, M, N), device=DEV)
    n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_STORE, y=z, ldy=N, kslices=slices)
    look(stamped(lambda: n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_STORE, y=y, ldy=N, kslices=slices)), workgroups)
    assert torch.equal(y, z)


@pytest.mark.parametrize("M", [5, 20])
@pytest.mark.parametrize("N,K", [(12288, 1120), (13824, 4096)])           # three and five tiles a workgroup
def test_epilogues(M, N, K):
    """A traced kernel stands for several epilogues: the sum into rows and the activation leave what their own kernels leave."""
    n = _n()
    wf, hi, lo, _ = operands(M, N, K)
    y, z = torch.ones((M, N), device=DEV), torch.ones((M, N), device=DEV)
    n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_ADD, y=z, ldy=N)
    assert stamped(lambda: n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_ADD, y=y, ldy=N)).shape[0] >= 173
    assert torch.equal(y, z)
    frags = [torch.zeros(((M + 15) // 16, N // 32, 64, 8), dtype=torch.float16, device=DEV) for _ in range(4)]
    n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_GELU, of_hi=frags[0], of_lo=frags[1])
    stamped(lambda: n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_GELU, of_hi=frags[2], of_lo=frags[3]))
    assert torch.equal(frags[0], frags[2]) and torch.equal(frags[1], frags[3]) and bool(frags[0].any())


# five tiles a workgroup only where they are the faster: images of 64 KB (up to 16 rows) and 128 KB, more than 840 tiles
@pytest.mark.parametrize("M,K,tiles,each", [(5, 4096, 1024, 5), (20, 4096, 841, 5), (32, 4096, 864, 5), (20, 4096, 832, 4), (12, 4096, 800, 4), (12, 2048, 1024, 5), (20, 2048, 1024, 4),
                                            (12, 6144, 1000, 4), (20, 8192, 1000, 4), (12, 4128, 1000, 4)])
def test_five_tiles_a_workgroup(M, K, tiles, each):
    n, N = _n(), 16 * tiles
    wf, hi, lo, want = operands(M, N, K)
    y = torch.zeros((M, N), device=DEV)
    look(stamped(lambda: n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_STORE, y=y, ldy=N)), -(-tiles // each))
    assert float((y.double() - want).norm() / want.norm()) < 1e-6
