"""pb_linear's tiles of 192 columns (bf16, many rows) against float64: 128 and 256 rows a tile, rows and columns that no tile divides, every way a result
leaves, activations of results that are rounded to bf16 and of those that are not."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64
BF = torch.bfloat16


def B():
    from promptcache_amd import _blocks
    return _blocks


def rnd(*shape, seed=0, dtype=BF):
    return torch.randn(*shape, generator=torch.Generator(device=DEV).manual_seed(seed), device=DEV).to(dtype)


def rel(got, want):
    return float((got.to(F64) - want).norm() / want.norm())


# fp32 results: a few hundred additions of exact products; bf16: half a last place, 2^-9 of each at most (2^-9 in the norm, less in fact)
@pytest.mark.parametrize("M,N,K", [(1000, 5133, 192), (4091, 2557, 192), (1003, 5136, 200)])          # 128 x 192, 256 x 192, k of no whole K-step
def test_every_way_out(M, N, K):
    b, f, low = B(), lambda t: t.to(F64), 2.0 ** -9
    x, w, bias = rnd(M, K, seed=1), rnd(N, K, seed=2) * 0.1, rnd(N, seed=3)
    z = f(x) @ f(w).T
    y = torch.full((M + 1, N), 7.0, device=DEV)
    b.linear(x, w, y, M=M)
    assert rel(y[:M], z) < 1e-6 and bool((y[M] == 7.0).all())
    rows = torch.randperm(M + 2, generator=torch.Generator().manual_seed(4))[:M].to(DEV, torch.int32)
    out = torch.zeros(M + 2, N, dtype=BF, device=DEV)
    for act, fn in ((b.ACT_SIGMOID, torch.sigmoid), (b.ACT_SILU, torch.nn.functional.silu)):
        b.linear(x, w, out, M=M, bias=bias, row_dst=rows, act_split=N // 3, act2=act)
        want = z + f(bias)
        want[:, N // 3:] = fn(want[:, N // 3:])
        assert rel(out[rows.long()], want) < low
        b.linear(x, w, y, M=M, bias=bias, act=act)                   # (fp32 results: as exact as they were)
        assert rel(y[:M], fn(z + f(bias))) < 1e-6
    split, cap = N - 256, M + 3
    first, heads = torch.empty(M, split, dtype=BF, device=DEV), torch.zeros(2, cap, 128, dtype=BF, device=DEV)
    b.linear(x, w, first, M=M, split_n=split, y2=heads, row_off2=(rows.long() * 128).contiguous(), head_dim2=128, head_stride2=cap * 128)
    assert rel(first, z[:, :split]) < low and rel(heads[:, rows.long()].transpose(0, 1).reshape(M, 256), z[:, split:]) < low
    base, scale = rnd(M, N, seed=6, dtype=torch.float32), rnd(N, seed=7, dtype=torch.float32)
    b.linear(x, w, y, M=M, epilogue=b.EPI_SCALE_ADD, bias=bias, base=base, col_scale=scale)
    assert rel(y[:M], f(base) + f(scale) * (z + f(bias))) < 1e-6
