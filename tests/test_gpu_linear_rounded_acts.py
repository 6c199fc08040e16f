"""Sigmoid and silu at the end of pb_linear's many-row tiles where results are rounded to bf16: against float64 over their range, at its ends, for infinities
and what is no number."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64
BF = torch.bfloat16


def B():
    from promptcache_amd import _blocks
    return _blocks


def test_activations_at_their_ends():
    b, M, N, K = B(), 1000, 5136, 64
    x, w = torch.zeros(M, K, device=DEV, dtype=BF), torch.zeros(N, K, device=DEV, dtype=BF)
    ends = [0.0, 1.0, -1.0, 20.0, -20.0, 60.0, -60.0, 100.0, -100.0, float("inf"), -float("inf"), float("nan")]
    bias = torch.tensor([ends[i % len(ends)] for i in range(N)], device=DEV).to(BF)
    out = torch.empty(M, N, dtype=BF, device=DEV)
    v = bias.to(F64)
    for act, want in ((b.ACT_SIGMOID, torch.sigmoid(v)), (b.ACT_SILU, v * torch.sigmoid(v))):
        b.linear(x, w, out, M=M, bias=bias, act=act)
        got = out[0].to(F64)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and bool((out[1:] == out[0]).eq(~torch.isnan(out[0])).all())
        fine = torch.isfinite(want)
        assert float((got[fine] - want[fine]).abs().max() / 1.0) < 60 * 2.0 ** -8 and float(((got - want).abs() / want.abs().clamp(min=1e-30))[fine].max()) < 2.0 ** -7
        inf = torch.isinf(want)
        assert torch.equal(got[inf], want[inf])
