"""Sigmoid and silu at the end of pb_linear's many-row tiles, as activations and as the gated unit: against float64 over their range, on both sides of where
the short form of the exponential ends, at their ends, for infinities and what is no number; results rounded to bf16 and in fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64
BF = torch.bfloat16


def B():
    from promptcache_amd import _blocks
    return _blocks


# an exponential good to a last place, a sum, a quotient: 2^-22 (measured 1.8e-7).  Rounded to bf16 half a last place more: neighbouring numbers of
# [1, 2) are 2^-7 apart, so 2^-8 of the value at most.
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2.0 ** -22), (BF, 2.0 ** -8 + 2.0 ** -22)])
@pytest.mark.parametrize("kind", ["sigmoid", "silu", "gated"])
def test_activations_over_their_range(kind, dtype, tol):
    b, M, N, K = B(), 1000, 5136, 64
    x, w = torch.zeros(M, K, device=DEV, dtype=BF), torch.zeros(N, K, device=DEV, dtype=BF)
    ends = [0.0, 20.0, -20.0, 60.0, -60.0, 86.5, -86.5, 87.0, -87.0, 87.5, -87.5, 100.0, -100.0, float("inf"), -float("inf"), float("nan")]
    v = torch.linspace(-20, 20, N, device=DEV)
    v[::5] = torch.linspace(-90, 90, len(v[::5]), device=DEV)
    v[7::321] = torch.tensor(ends, device=DEV)[:len(v[7::321])]
    bias = v.to(BF)
    v, out = bias.to(F64), torch.empty(M, N, dtype=dtype, device=DEV)
    want = torch.sigmoid(v) if kind == "sigmoid" else v * torch.sigmoid(v)
    if kind == "gated":
        b.linear(x, w, out, M=M, bias=bias, epilogue=b.EPI_SILU_MUL, w2=w, bias2=torch.full((N,), 2.0, device=DEV, dtype=BF))
        want = 2 * want
    else:
        b.linear(x, w, out, M=M, bias=bias, act=b.ACT_SIGMOID if kind == "sigmoid" else b.ACT_SILU)
    assert bool(((out == out[0]) | torch.isnan(out[0])).all())
    got, fine = out[0].to(F64), torch.isfinite(want)
    assert int((~fine).sum()) >= (1 if kind == "sigmoid" else 3) and torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf], want[inf])
    # (below -88.7 the exponential is infinity and results are 0, where 2 |v| e^v is below 2^-119)
    assert bool(((got - want).abs()[fine] <= (tol * want.abs()[fine]).clamp(min=2.0 ** -119)).all())
