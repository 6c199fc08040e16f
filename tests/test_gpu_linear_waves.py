"""pb_linear over some tens or hundreds of rows against float64: rows and columns that no tile of 32 divides, k of less than a chunk, of fewer chunks than
waves and of none to a whole number of them, the borders of the rule (256, 512, 768 workgroups), and every way a result leaves."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


def B():
    from promptcache_amd import _blocks
    return _blocks


def rnd(*shape, seed=0, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV, dtype)


def rel(got, want):
    return float((got.to(F64) - want).norm() / want.norm())


# sums of up to 4096 exact or once rounded products in a few hundred fp32 additions each: 1e-6; bf16 results add half a last place, 2^-8 at most
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(17, 36, 8), (31, 1001, 96), (33, 70, 200), (64, 1024, 1024), (37, 512, 4096), (130, 1030, 1152), (100, 2051, 264),
                                   (256, 1024, 512), (257, 1024, 2048), (512, 1024, 1024), (513, 1024, 512), (600, 1024, 1024), (769, 1024, 2048)])
def test_every_way_out(M, N, K, dtype):
    b, f = B(), lambda t: t.to(F64)
    low = 1e-6 if dtype == torch.float32 else 2.0 ** -8
    x, w, bias = rnd(M + 2, K, seed=1, dtype=dtype), rnd(N, K, seed=2, dtype=dtype) * 0.1, rnd(N, seed=3, dtype=dtype)
    rows = torch.randperm(M + 2, generator=torch.Generator().manual_seed(4))[:M].to(DEV, torch.int32)
    z = f(x)[:M] @ f(w).T
    y = torch.full((M + 1, N), 7.0, device=DEV)
    b.linear(x, w, y, M=M)
    assert rel(y[:M], z) < 1e-6 and bool((y[M] == 7.0).all())
    # gathered and scattered rows, bias, a sigmoid from a column on
    split, out = N // 3 + 1, torch.zeros(M + 2, N, dtype=dtype, device=DEV)
    b.linear(x, w, out, M=M, bias=bias, row_src=rows, row_dst=rows, act_split=split, act2=b.ACT_SIGMOID)
    want = f(x)[rows.long()] @ f(w).T + f(bias)
    want[:, split:] = want[:, split:].sigmoid()
    assert rel(out[rows.long()], want) < low
    # columns split off to a cache's heads of four columns, rows where a table says
    first, cap, heads = torch.empty(M, N - 8, dtype=dtype, device=DEV), M + 3, torch.zeros(2, M + 3, 4, dtype=dtype, device=DEV)
    off = (rows.long() * 4).contiguous()
    b.linear(x, w, first, M=M, split_n=N - 8, y2=heads, row_off2=off, head_dim2=4, head_stride2=cap * 4)
    assert rel(first, z[:, :N - 8]) < low and rel(heads[:, rows.long()].transpose(0, 1).reshape(M, 8), z[:, N - 8:]) < low
    # gated unit
    w2, gate = rnd(N, K, seed=5, dtype=dtype) * 0.1, rnd(M, 3, seed=8, dtype=dtype)
    mid = torch.empty(M, N, dtype=dtype, device=DEV)
    b.linear(x, w, mid, M=M, epilogue=b.EPI_SILU_MUL, w2=w2, bias=bias, row_gate=gate, ld_row_gate=3)
    assert rel(mid, torch.nn.functional.silu(z + f(bias)) * (f(x)[:M] @ f(w2).T) * f(gate)[:, :1]) < max(low, 2e-6)
    # scaled accumulation, onto another matrix and in place
    base, scale = rnd(M, N, seed=6), rnd(N, seed=7)
    b.linear(x, w, y, M=M, epilogue=b.EPI_SCALE_ADD, bias=bias, base=base, col_scale=scale)
    want = f(base) + f(scale) * (z + f(bias))
    assert rel(y[:M], want) < 1e-6
    b.linear(x, w, y, M=M, epilogue=b.EPI_SCALE_ADD, col_scale=scale)
    assert rel(y[:M], want + f(scale) * z) < 1e-6 and bool((y[M] == 7.0).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,n", [(20, 36, 64, 3), (75, 128, 192, 16), (300, 40, 512, 2)])
def test_batches(M, N, K, n, dtype):
    x, w = rnd(M, n * K, seed=1, dtype=dtype), rnd(n, N, K, seed=2, dtype=dtype)
    y = torch.empty(M, n * N, device=DEV)
    B().linear(x, w, y, M=M, n_batch=n, ldx=n * K, x_batch_stride=K, ldy=n * N, y_batch_stride=N)
    want = torch.stack([x.to(F64)[:, i * K:(i + 1) * K] @ w[i].to(F64).T for i in range(n)], 1).reshape(M, n * N)
    assert rel(y, want) < 1e-6


def test_a_row_that_is_no_number_stays_alone():
    b, M, N, K = B(), 40, 64, 512
    x, w, y = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, dtype=torch.bfloat16), torch.empty(M, N, device=DEV)
    b.linear(x, w, y, M=M)
    clean, x = y.clone(), x.clone()
    x[9, 100] = float("nan")
    b.linear(x, w, y, M=M)
    keep = [r for r in range(M) if r != 9]
    assert bool(torch.isnan(y[9]).all()) and torch.equal(y[keep], clean[keep])
