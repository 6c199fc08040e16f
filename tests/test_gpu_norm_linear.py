"""The residual row, its norm and the products of the normed rows in one launch (pb_linear_normed.hip), against torch in 64 bits and the launches it stands for."""
import pytest
import torch

from promptcache_amd import _blocks as B

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rms(x, gain, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gain


def rand(*shape, dtype=torch.float32, sd=1.0, seed=[0]):
    seed[0] += 1
    g = torch.Generator().manual_seed(seed[0])
    return (torch.randn(*shape, generator=g) * sd).to(dtype).to(DEV)


CASES = [  # (rows, k, columns, of the second product): whole and odd tiles of columns; last k-steps of no wave, one, all; chunks, rows and runs at their edges
    (1, 64, 8, 0), (1, 512, 40, 24), (2, 512, 100, 33), (3, 512, 33, 0), (4, 512, 64, 130), (5, 256, 70, 18), (8, 512, 48, 31), (1, 576, 96, 17), (1, 1024, 48, 56),
    (2, 1024, 72, 9), (3, 1024, 33, 40), (4, 1024, 24, 64), (1, 1088, 80, 30), (1, 2048, 56, 41), (2, 1024, 1600, 700), (1, 1024, 5000, 0), (1, 2048, 4000, 1700)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["table", "mix1", "mix3", "mix7", "mix11", "post", "gated"])
@pytest.mark.parametrize("M,K,N1,N2", CASES)
def test_norm_linear(dtype, kind, M, K, N1, N2):
    N2 = N2 or (24 if kind == "gated" else 0)                        # (the gated unit is the second product)
    fp32 = dtype == torch.float32
    gain, gain2, post = (rand(K, sd=0.1) + 1 for _ in range(3))
    w1, b1 = rand(N1, K, dtype=dtype, sd=K ** -0.5), rand(N1, dtype=dtype, sd=0.1)
    h1, h2, xo = torch.empty(M, K, dtype=dtype, device=DEV), torch.empty(M, K, dtype=dtype, device=DEV), torch.full((M, K), 9.0, device=DEV)
    split = kind.startswith("mix") and N1 % 8 == 0 and N1 > 8       # columns from here on into rows of a cache, heads of four or eight columns
    heads = 8 if N1 % 16 == 0 else 4
    y1 = torch.full((M, N1 // 2 // 4 * 4 if split else N1), 7.0, dtype=dtype, device=DEV)
    s = y1.shape[1]
    cache, off = torch.full((9, 2 * N1), 7.0, dtype=dtype, device=DEV), torch.tensor([2 * N1 * ((3 * m + 1) % 8) for m in range(M)], dtype=torch.int64, device=DEV)
    kw = dict(split_n=s, y2=cache, row_off2=off, head_dim2=heads if (N1 - s) % heads == 0 else 4, head_stride2=12) if split else \
        dict(act_split=max(4, N1 // 3), act2=B.ACT_SIGMOID)
    a = B.linear_args(h1, w1, y1, M=M, bias=b1, **kw)
    b = None
    if N2:
        w2, b2 = rand(N2, K, dtype=dtype, sd=K ** -0.5), rand(N2, dtype=dtype, sd=0.1)
        if kind == "gated":
            w3, b3 = rand(N2, K, dtype=dtype, sd=K ** -0.5), rand(N2, dtype=dtype, sd=0.1)
            y2 = torch.full((M, N2), 7.0, dtype=dtype, device=DEV)
            b = B.linear_args(h1, w2, y2, M=M, epilogue=B.EPI_SILU_MUL, w2=w3, bias=b2, bias2=b3)
        else:
            y2 = torch.full((M, N2), 7.0, device=DEV)
            b = B.linear_args(h2, w2, y2, M=M, bias=b2)
    d = torch.float64
    if kind == "table":
        table, ids = rand(50, K, dtype=dtype), torch.tensor([(7 * m + 49) % 53 for m in range(M)], dtype=torch.int32, device=DEV)
        src, x = dict(table=table, ids=ids, scale=1.5), 1.5 * table.to(d)[ids.clamp(0, 49).long()]
    elif kind.startswith("mix"):
        n = int(kind[3:])
        hist, coef = rand(n + 1, M, K), rand(n, sd=0.5)
        hist[n] = float("nan")                                       # (what lies behind the last stream is not counted)
        src, x = dict(x=hist, coef=coef, n_terms=n), torch.einsum("j,jmk->mk", coef.to(d), hist[:n].to(d))
    else:
        r, y, wide = rand(M, K), rand(M, K), torch.rand(M, K + 12, device=DEV).to(dtype)
        src, x = dict(x=r, y=y, gate=wide[:, 4:], ldg=K + 12, post_gain=post), r.to(d) + rms(y.to(d) * wide[:, 4:4 + K].to(d), post.to(d))
    taken = B.norm_linear(a, b, gain, (gain if kind == "gated" else gain2) if b else None, xo, eps=1e-5, **src)
    if not taken:                                                    # more columns than it is the faster one for: nothing done
        assert N1 >= 1600
        assert (xo == 9).all() and (y1 == 7).all() and (cache == 7).all() and (not N2 or (y2 == 7).all())
        return
    # the residual: a few fp32 roundings of terms of the sums' sizes
    assert (xo.to(d) - x).abs().max() <= 2e-6 * (1 + x.abs().max())
    # the products: fp32 roundings of the row and of sums over k; bf16: the row's rounding (2^-9 of each term, at random: sqrt(k) of terms k^-1/2) and the result's
    n1 = rms(x, gain.to(d))
    n2 = n1 if kind == "gated" else rms(x, gain2.to(d))

    def close(got, want):
        scale = n1.abs().max() if fp32 else 1.0
        tol = 4e-6 * scale * (1 + want.abs()) if fp32 else 2 ** -8 * want.abs() + 6 * 2 ** -9 * 1.5 * (1 + want.abs())
        assert ((got.to(d) - want).abs() <= tol).all(), ((got.to(d) - want).abs() / tol).max()

    want = n1 @ w1.to(d).T + b1.to(d)
    if split:
        close(y1, want[:, :s])
        got = torch.stack([torch.stack([cache.view(-1)[int(off[m]) + c // kw["head_dim2"] * 12 + c % kw["head_dim2"]] for c in range(N1 - s)]) for m in range(M)])
        close(got, want[:, s:])
        assert int((cache != 7).sum()) <= M * (N1 - s)
    else:
        want[:, max(4, N1 // 3):] = torch.sigmoid(want[:, max(4, N1 // 3):])
        close(y1, want)
    if N2:
        want = n2 @ w2.to(d).T + b2.to(d)
        if kind == "gated":
            want = torch.nn.functional.silu(want) * (n2 @ w3.to(d).T + b3.to(d))
        close(y2, want)
    # the launches that it stands for
    h, hh, x2 = torch.empty_like(h1), torch.empty_like(h1), torch.empty_like(xo)
    if kind == "table":
        B.embed_scaled_rows(table, ids, 1.5, x2)
        B.post_norm(x2, gain=gain, out=h, eps=1e-5, n_rows=M)
    elif kind.startswith("mix"):
        B.mix_norm(hist, n, coef, gain, h, gain2, hh, x_out=x2, eps=1e-5, n_rows=M)
    else:
        x2.copy_(r)
        B.post_norm(x2, gain=gain, out=h, eps=1e-5, n_rows=M, y=y, gate=wide[:, 4:], ldg=K + 12, post_gain=post)
    assert (x2 - xo).abs().max() <= 1e-6 * (1 + x2.abs().max())
    if not split:
        z = torch.empty_like(y1)
        B.linear(h, w1, z, M=M, bias=b1, **kw)
        close(y1, z.to(d))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,W", [(1, 4), (3, 260), (2, 2048), (700, 1024), (1, 8192), (5, 16384), (4, 1001), (513, 512)])
@pytest.mark.parametrize("both", [False, True])
def test_embed_norm(dtype, rows, W, both):
    table, ids = rand(40, W, dtype=dtype), torch.tensor([(11 * r + 41) % 45 - 2 for r in range(rows)], dtype=torch.int32, device=DEV)
    g1, g2 = rand(W, sd=0.1) + 1, rand(W, sd=0.1) + 1
    x, o1, o2 = torch.empty(rows, W, device=DEV), torch.empty(rows, W, dtype=dtype, device=DEV), torch.empty(rows, W, dtype=dtype, device=DEV)
    B.embed_norm(table, ids, 0.75, x, g1, o1, g2 if both else None, o2 if both else None, eps=1e-5)
    want = 0.75 * table.float()[ids.clamp(0, 39).long()]
    assert torch.equal(x, want)
    for g, o in ((g1, o1), (g2, o2))[:1 + both]:
        n = rms(want.double(), g.double())
        # (fp32: a sum of squares, a root, a quotient and two products; bf16: the result's rounding)
        assert ((o.double() - n).abs() <= (2.0 ** -21 if dtype == torch.float32 else 2.0 ** -8) * n.abs() + 1e-30).all()
