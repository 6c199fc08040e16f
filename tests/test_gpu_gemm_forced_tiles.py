"""PC_GEMM_T, the number of tiles a workgroup that probes force: every launch still has a kernel (fewer tiles where there is none of so many) and the right sums."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CODE = """
import torch
from tests.test_gpu_gemm_pipe import operands
from tests.test_gpu_gemm_norm import EPS, exact, inputs
from promptcache_amd import _native as n
DEV = "cuda"
N, K = 4096, 288
for M in (1, 12, 20, 40, 64):
    wf, hi, lo, want = operands(M, N, K)
    for epi in (n.EPI_STORE, n.EPI_ADD):
        y = torch.zeros((M, N), device=DEV)
        n.gemm_skinny(wf, hi, lo, M, N, K, epi, y=y, ldy=N)
        assert float((y.double() - want).norm() / want.norm()) < 1e-6, (M, epi)
    oh = torch.zeros((hi.shape[0], N // 64, 64, 8), dtype=torch.float16, device=DEV)
    ol = torch.zeros_like(oh)
    n.gemm_skinny(wf, hi, lo, M, N, K, n.EPI_SILU, of_hi=oh, of_lo=ol)
    gated = torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:]
    got = n.from_act_frags(oh, M).double() + n.from_act_frags(ol, M).double()
    assert float((got - gated).norm() / gated.norm()) < 2e-6, M
    if M <= 16:
        w, x, gam = inputs(M, N, K)
        y = torch.zeros((M, N), device=DEV)
        n.gemm_skinny_norm(n.to_weight_frags(w), x, gam, EPS, M, N, K, n.EPI_STORE, y=y, ldy=N)
        want = exact(x, gam, w)
        assert float((y.double() - want).norm() / want.norm()) < 1e-6, M
print("all right")
"""


@pytest.mark.parametrize("tiles", [1, 5, 8])
def test_forced_tiles(tiles):
    env = dict(os.environ, PC_GEMM_T=str(tiles), PYTHONPATH=os.pathsep.join([ROOT, os.path.join(ROOT, "prompt-cache_amd")]))
    r = subprocess.run([sys.executable, "-c", CODE], cwd=ROOT, env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "all right" in r.stdout, r.stderr[-2000:]
