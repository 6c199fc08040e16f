"""pb_linear of up to sixteen rows against float64: row counts around the four, eight and sixteen rows of a product with its runs of k side by side,
column counts that no workgroup divides and that cross the borders of the rule, k of one k-step to several rounds of the waves, and every way a result
leaves (bias and activations, split columns, gathered and scattered rows, gated units, scaled accumulation, batches)."""
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


# products are exact or rounded once to fp32, sums of up to 4096 of them run in a few hundred fp32 additions each: 1e-6; bf16 results add half a last
# place, 2^-8 at most
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 3, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("N,K", [(20, 32), (1001, 512), (1030, 1024), (3077, 1152), (2056, 2048), (3300, 2176), (8200, 1024), (70, 4096)])
def test_few_rows(M, N, K, dtype):
    b, f = B(), lambda t: t.to(F64)
    low = 1e-6 if dtype == torch.float32 else 2.0 ** -8
    x, w, bias = rnd(M + 2, K, seed=1, dtype=dtype), rnd(N, K, seed=2, dtype=dtype) * 0.1, rnd(N, seed=3, dtype=dtype)
    rows = torch.randperm(M + 2, generator=torch.Generator().manual_seed(4))[:M].to(DEV, torch.int32)
    z = f(x)[:M] @ f(w).T
    y = torch.empty(M, N, device=DEV)
    b.linear(x, w, y, M=M)
    assert rel(y, z) < 1e-6
    # gathered and scattered rows, bias, a sigmoid from a column on
    split, out = N // 3 + 1, torch.zeros(M + 2, N, dtype=dtype, device=DEV)
    b.linear(x, w, out, M=M, bias=bias, row_src=rows, row_dst=rows, act_split=split, act2=b.ACT_SIGMOID)
    want = f(x)[rows.long()] @ f(w).T + f(bias)
    want[:, split:] = want[:, split:].sigmoid()
    assert rel(out[rows.long()], want) < low
    # columns split off to a second matrix
    first, second = torch.empty(M, split, dtype=dtype, device=DEV), torch.zeros(M, N - split, device=DEV)
    b.linear(x, w, first, M=M, split_n=split, y2=second, y2_f32=True, head_stride2=N - split)
    assert rel(first, z[:, :split]) < low and rel(second, z[:, split:]) < 1e-6
    # gated unit
    w2 = rnd(N, K, seed=5, dtype=dtype) * 0.1
    mid = torch.empty(M, N, dtype=dtype, device=DEV)
    b.linear(x, w, mid, M=M, epilogue=b.EPI_SILU_MUL, w2=w2, bias=bias)
    assert rel(mid, torch.nn.functional.silu(z + f(bias)) * (f(x)[:M] @ f(w2).T)) < max(low, 2e-6)
    # scaled accumulation onto another matrix
    base, scale = rnd(M, N, seed=6), rnd(N, seed=7)
    b.linear(x, w, y, M=M, epilogue=b.EPI_SCALE_ADD, bias=bias, base=base, col_scale=scale)
    assert rel(y, f(base) + f(scale) * (z + f(bias))) < 1e-6


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,n", [(2, 36, 1024, 5), (8, 24, 512, 16), (13, 40, 96, 3)])
def test_few_rows_of_a_batch(M, N, K, n, dtype):
    x, w = rnd(M, n * K, seed=1, dtype=dtype), rnd(n, N, K, seed=2, dtype=dtype)
    y = torch.empty(M, n * N, device=DEV)
    B().linear(x, w, y, M=M, n_batch=n, ldx=n * K, x_batch_stride=K, ldy=n * N, y_batch_stride=N)
    want = torch.stack([x.to(F64)[:, i * K:(i + 1) * K] @ w[i].to(F64).T for i in range(n)], 1).reshape(M, n * N)
    assert rel(y, want) < 1e-6


# sizes on both sides of the rule's other borders: one run late and not, a deep k of few and of many columns, four runs' and two runs' last sizes
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [2, 4, 7, 12])
@pytest.mark.parametrize("N,K", [(12300, 64), (12300, 96), (8250, 480), (8200, 512), (8200, 1024), (6200, 960), (2600, 4096), (4100, 4096), (8300, 4096)])
def test_few_rows_at_the_rules_other_borders(M, N, K, dtype):
    b, f = B(), lambda t: t.to(F64)
    low = 1e-6 if dtype == torch.float32 else 2.0 ** -8
    x, w, w2 = rnd(M, K, seed=1, dtype=dtype), rnd(N, K, seed=2, dtype=dtype) * 0.1, rnd(N, K, seed=5, dtype=dtype) * 0.1
    z, out, y = f(x) @ f(w).T, torch.empty(M, N, dtype=dtype, device=DEV), rnd(M, N, seed=6)
    b.linear(x, w, out, M=M)
    assert rel(out, z) < low
    b.linear(x, w, out, M=M, epilogue=b.EPI_SILU_MUL, w2=w2, act=b.ACT_RELU)
    assert rel(out, z.relu() * (f(x) @ f(w2).T)) < max(low, 2e-6)
    scale, want = rnd(N, seed=7), f(y)
    b.linear(x, w, y, M=M, epilogue=b.EPI_SCALE_ADD, col_scale=scale)
    assert rel(y, want + f(scale) * z) < 1e-6


# several blocks of eight columns a workgroup: a block more than a round of the chip, last workgroups of one block or a part of it, two, three and four blocks, k of
# one, two and three trips, weights read past the caches (rows of 4 KB, 4 MB) and not
@pytest.mark.parametrize("M", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("N,K", [(2049, 1024), (4609, 1088), (6144, 1984), (8161, 2048), (8193, 2112), (6137, 4096), (16385, 1024)])
def test_several_blocks_of_columns_a_workgroup(M, N, K):
    b, f, dtype = B(), lambda t: t.to(F64), torch.bfloat16
    x, w, bias = rnd(M, K, seed=1, dtype=dtype), rnd(N, K, seed=2, dtype=dtype) * 0.1, rnd(N, seed=3, dtype=dtype)
    out, y, z = torch.zeros(M + 1, N, dtype=dtype, device=DEV), torch.empty(M, N, device=DEV), f(x) @ f(w).T
    b.linear(x, w, y, M=M)
    assert rel(y, z) < 1e-6
    b.linear(x, w, out, M=M, bias=bias, act_split=N // 3, act2=b.ACT_SIGMOID)
    want = z + f(bias)
    want[:, N // 3:] = want[:, N // 3:].sigmoid()
    assert rel(out[:M], want) < 2.0 ** -8 and not bool(out[M].any())
