"""Two products in one launch (pcb_linear_pair, pcb_linear_add2) against the launches that they stand for and against float64: row counts around the one,
two, four and eight rows of a runs' product and beyond, columns that no workgroup divides, k of a few and of many steps, what falls back."""
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


# fp32 sums of up to 4096 products in a few hundred additions each: 1e-6; bf16 results half a last place more, 2^-8 at most
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 2, 4, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("N,N2,K,K2", [(1280, 4096, 1024, 1024), (37, 1001, 96, 512), (1026, 20, 2048, 1088), (5000, 5000, 1024, 1024), (64, 64, 1024, 40)])
def test_pairs(M, N, N2, K, K2, dtype):
    b, f = B(), lambda t: t.to(F64)
    low = 1e-6 if dtype == torch.float32 else 2.0 ** -8
    x, x2, w, v, v2 = (rnd(*s, seed=i, dtype=dtype) for i, s in enumerate([(M, K), (M, K2), (N, K), (N2, K2), (N2, K2)]))
    bias = rnd(N, seed=9, dtype=dtype)
    first, plane, z = torch.empty(M, N // 2, dtype=dtype, device=DEV), torch.zeros(M, N - N // 2, device=DEV), torch.empty(M, N2, device=DEV)
    b.linear_pair(b.linear_args(x, w, first, M=M, bias=bias, split_n=N // 2, y2=plane, y2_f32=True, head_stride2=N - N // 2), b.linear_args(x2, v, z, M=M))
    want = f(x) @ f(w).T + f(bias)
    assert rel(first, want[:, :N // 2]) < low and rel(plane, want[:, N // 2:]) < 1e-6 and rel(z, f(x2) @ f(v).T) < 1e-6
    gate, mid = torch.empty(M, N, dtype=dtype, device=DEV), torch.empty(M, N2, dtype=dtype, device=DEV)
    b.linear_pair(b.linear_args(x, w, gate, M=M, bias=bias, act=b.ACT_SIGMOID),
                  b.linear_args(x2, v, mid, M=M, epilogue=b.EPI_SILU_MUL, w2=v2, act=b.ACT_RELU))
    assert rel(gate, want.sigmoid()) < max(low, 2e-6) and rel(mid, (f(x2) @ f(v).T).relu() * (f(x2) @ f(v2).T)) < max(low, 2e-6)


# two blocks of the first product's columns a workgroup (a round of the chip less), the last one of a part of a block; k of one product beyond the line, of the other not
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 5, 8])
@pytest.mark.parametrize("N,N2,K,K2", [(1540, 3070, 1536, 1536), (1537, 3072, 1600, 1088), (3000, 9, 1088, 1024)])
def test_pairs_beside_a_gated_unit_of_two_runs(M, N, N2, K, K2, dtype):
    test_pairs(N=N, N2=N2, K=K, K2=K2, M=M, dtype=dtype)


# either side of the lines between one run and two: 1024 of k (results' places ahead), just more and just fewer, 7168 weight rows of a gated unit and 8192 plain ones, in fp32 16384 over 1024
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [4, 5, 8])
@pytest.mark.parametrize("N,N2,K,K2", [(1024, 3072, 1024, 1024), (1024, 3073, 1024, 1088), (1040, 3064, 512, 512), (1040, 3065, 512, 960), (2048, 7168, 1024, 1024), (2048, 7170, 1024, 1024),
                                       (1024, 3072, 1472, 1472), (1025, 7168, 1536, 1600)])
def test_pairs_on_either_side_of_the_lines(M, N, N2, K, K2, dtype):
    test_pairs(N=N, N2=N2, K=K, K2=K2, M=M, dtype=dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M", [1, 2, 3, 5, 8, 9])
@pytest.mark.parametrize("N,K,ff", [(1024, 1024, 4096), (1001, 512, 1536), (70, 1152, 512), (36, 64, 96)])
def test_two_accumulations(M, N, K, ff, dtype):
    b, f = B(), lambda t: t.to(F64)
    x, w, v, bias = rnd(M, K, seed=1, dtype=dtype), rnd(N, K, seed=2, dtype=dtype), rnd(N, ff, seed=3, dtype=dtype), rnd(N, seed=4, dtype=dtype)
    base, s1, s2, z, coef = rnd(M, N, seed=5), rnd(N, seed=6), rnd(N, seed=7), rnd(M, ff, seed=8) + 0.3, rnd(4, seed=9)
    act, y = torch.zeros(M, ff, dtype=dtype, device=DEV), torch.zeros(M, N, device=DEV)

    def both(**kw):
        b.linear_add2(b.linear_args(x, w, y, M=M, epilogue=b.EPI_SCALE_ADD, bias=bias, base=base, col_scale=s1),
                      b.linear_args(act, v, y, M=M, epilogue=b.EPI_SCALE_ADD, col_scale=s2), **kw)
        return y.clone()
    first = f(base) + f(s1) * (f(x) @ f(w).T + f(bias))
    got = both(z=z, coef=coef, eps=1e-6)
    b.polynorm(z, coef, act, 1e-6, M)
    want = first + f(s2) * (f(act) @ f(v).T)
    # (inputs that a launch of its own would round to the neighbouring bf16 number: a few of them, half a last place each)
    assert rel(got, want) < (2e-6 if dtype == torch.float32 else 1e-4)
    assert rel(both(), want) < 1e-6


def test_a_row_that_is_no_number_stays_alone():
    b, M, N, K, ff = B(), 3, 1024, 1024, 4096
    x, w, v, z = rnd(M, K, dtype=torch.bfloat16), rnd(N, K, seed=1, dtype=torch.bfloat16), rnd(N, ff, seed=2, dtype=torch.bfloat16), rnd(M, ff, seed=3)
    act, y, one = torch.zeros(M, ff, dtype=torch.bfloat16, device=DEV), torch.zeros(M, N, device=DEV), torch.ones(N, device=DEV)

    def run(z):
        y.zero_()
        b.linear_add2(b.linear_args(x, w, y, M=M, epilogue=b.EPI_SCALE_ADD, col_scale=one),
                      b.linear_args(act, v, y, M=M, epilogue=b.EPI_SCALE_ADD, col_scale=one), z, rnd(4, seed=4), 1e-6)
        return y.clone()
    clean, bad = run(z), z.clone()
    bad[1, 7] = float("nan")
    got = run(bad)
    assert bool(torch.isnan(got[1]).all()) and torch.equal(got[[0, 2]], clean[[0, 2]])


def test_what_is_refused():
    b = B()
    x, w, y = rnd(2, 64), rnd(32, 64), torch.zeros(2, 32, device=DEV)
    s = torch.ones(32, device=DEV)
    add = b.linear_args(x, w, y, M=2, epilogue=b.EPI_SCALE_ADD, col_scale=s)
    for other in (b.linear_args(x, w, y, M=2), b.linear_args(x, w, torch.zeros(2, 32, device=DEV), M=2, epilogue=b.EPI_SCALE_ADD, col_scale=s),
                  b.linear_args(x, w, y, M=1, epilogue=b.EPI_SCALE_ADD, col_scale=s)):
        with pytest.raises(RuntimeError, match="same rows"):
            b.linear_add2(add, other)
