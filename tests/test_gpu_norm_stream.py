"""The norm in the launch of its products with one workgroup a CU (pcb_norm_stream) against torch in 64 bits and the launches that it stands for."""
import pytest
import torch

from promptcache_amd import _blocks as B

pytestmark = pytest.mark.gpu
DEV = "cuda"

# rows, k, columns, of the second product: fewer blocks of eight columns than CUs and more, one left over, odd last blocks; k-steps of no, some and all waves; 1 to 8 chunks of a row
CASES = [(1, 576, 9, 0), (2, 1024, 2048, 40), (3, 640, 2057, 0), (4, 1024, 4100, 13), (5, 832, 31, 3000), (8, 1024, 6151, 0), (1, 1600, 8, 24), (2, 2048, 50, 0), (3, 1984, 700, 1031),
         (4, 2048, 2048, 2056), (6, 1664, 2049, 0), (8, 2048, 33, 17), (7, 2048, 6200, 0), (8, 2048, 1029, 2100)]


def rms(x, gain, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * gain


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("kind", ["table", "mix1", "mix2", "mix5", "post", "gated"])
@pytest.mark.parametrize("M,K,N1,N2", CASES)
def test_norm_stream(dtype, kind, M, K, N1, N2):
    g = torch.Generator().manual_seed(M * K + N1)
    rand = lambda *s, sd=1.0, dt=torch.float32: (torch.randn(*s, generator=g) * sd).to(dt).to(DEV)       # noqa: E731
    d, fp32 = torch.float64, dtype == torch.float32
    N2 = N2 or (24 if kind == "gated" else 0)
    gain, post = rand(K, sd=0.1) + 1, rand(K, sd=0.1) + 1
    gain2 = gain if kind in ("gated", "mix5") else rand(K, sd=0.1) + 1
    w, bias = rand(N1, K, sd=K ** -0.5, dt=dtype), rand(N1, sd=0.1, dt=dtype)
    h = torch.empty(M, K, dtype=dtype, device=DEV)
    cut = N1 // 2 if kind == "mix2" and N1 % 16 == 8 else 0         # (columns from here on into rows of a cache, heads of four)
    y = torch.full((M + 1, cut or N1), 7.0, dtype=dtype, device=DEV)
    cache, off = torch.full((M, 3 * N1), 7.0, dtype=dtype, device=DEV), torch.tensor([3 * N1 * (M - 1 - m) for m in range(M)], dtype=torch.int64, device=DEV)
    kw = dict(split_n=cut, y2=cache, row_off2=off, head_dim2=4, head_stride2=8) if cut else dict(act_split=max(1, N1 // 3), act2=B.ACT_SIGMOID)
    a, b = B.linear_args(h, w, y, M=M, bias=bias, **kw), None
    y2 = torch.full((M + 1, max(N2, 1)), 7.0, dtype=dtype if kind == "gated" else torch.float32, device=DEV)
    if N2:
        w2, w3, b2, b3 = rand(N2, K, sd=K ** -0.5, dt=dtype), rand(N2, K, sd=K ** -0.5, dt=dtype), rand(N2, sd=0.1, dt=dtype), rand(N2, sd=0.1, dt=dtype)
        b = B.linear_args(h, w2, y2, M=M, epilogue=B.EPI_SILU_MUL, w2=w3, bias=b2, bias2=b3) if kind == "gated" else B.linear_args(h, w2, y2, M=M, bias=b2)
    if kind == "table":
        table, ids = rand(50, K, dt=dtype), torch.tensor([(7 * m + 49) % 53 for m in range(M)], dtype=torch.int32, device=DEV)
        src, x = dict(table=table, ids=ids, scale=1.5), 1.5 * table.to(d)[ids.clamp(0, 49).long()]
    elif kind.startswith("mix"):
        n = int(kind[3:])
        hist, coef = rand(n + 1, M, K), rand(n, sd=0.5)
        hist[n] = float("nan")                                       # (behind the last stream: not counted)
        src, x = dict(x=hist, coef=coef, n_terms=n), torch.einsum("j,jmk->mk", coef.to(d), hist[:n].to(d))
    else:
        r, t, wide = rand(M, K), rand(M, K), torch.rand(M, K + 12, generator=g).to(dtype).to(DEV)
        src, x = dict(x=r, y=t, gate=wide[:, 4:], ldg=K + 12, post_gain=post), r.to(d) + rms(t.to(d) * wide[:, 4:4 + K].to(d), post.to(d), 1e-5)
    xo = torch.full((M + 1, K), 9.0, device=DEV)
    elems = K << (0 if M == 1 else 1 if M == 2 else 2 if M <= 4 else 3)
    runs = -(-N1 // 8) + -(-N2 // 8)
    taken = B.norm_linear(a, b, gain, gain2 if b else None, xo, eps=1e-5, many=True, **src)
    assert taken == (not kind.startswith("mix") or n * elems <= (32768 if runs > 256 else 12288))
    assert (xo[M:] == 9).all() and (y[M:] == 7).all() and (y2[M:] == 7).all()
    if not taken:                                                    # nothing done
        assert (xo == 9).all() and (y == 7).all() and (y2 == 7).all() and (cache == 7).all()
        return
    # the residual: a few fp32 roundings of terms of the sums' sizes
    assert (xo[:M].to(d) - x).abs().max() <= 2e-6 * (1 + x.abs().max())
    n1, n2 = rms(x, gain.to(d), 1e-5), rms(x, gain2.to(d), 1e-5)

    def close(got, want):
        # fp32: roundings of the row and of sums over k; bf16: the row's rounding (2^-9 of each term, at random: sqrt(k) of terms k^-1/2) and the result's
        tol = 4e-6 * n1.abs().max() * (1 + want.abs()) if fp32 else 2 ** -8 * want.abs() + 6 * 2 ** -9 * 1.5 * (1 + want.abs())
        assert ((got.to(d) - want).abs() <= tol).all(), ((got.to(d) - want).abs() / tol).max()

    want = n1 @ w.to(d).T + bias.to(d)
    if cut:
        close(y[:M], want[:, :cut])
        c = torch.arange(N1 - cut, device=DEV)
        at = off[:, None] + c // 4 * 8 + c % 4
        close(cache.view(-1)[at], want[:, cut:])
        assert int((cache != 7).sum()) <= M * (N1 - cut)
    else:
        want[:, max(1, N1 // 3):] = torch.sigmoid(want[:, max(1, N1 // 3):])
        close(y[:M], want)
    if N2:
        want = n2 @ w2.to(d).T + b2.to(d)
        close(y2[:M], torch.nn.functional.silu(want) * (n2 @ w3.to(d).T + b3.to(d)) if kind == "gated" else want)


# a vocabulary's columns of a short k, and many streams of one: whether the launch is taken, by type, rows and k
@pytest.mark.parametrize("dtype,kind,M,K,N,taken", [
    (torch.bfloat16, "post", 1, 896, 24008, False), (torch.bfloat16, "post", 1, 960, 24008, True), (torch.bfloat16, "post", 4, 704, 24008, False), (torch.bfloat16, "post", 3, 768, 24008, True),
    (torch.bfloat16, "post", 8, 640, 24008, False), (torch.bfloat16, "post", 5, 704, 24008, True), (torch.bfloat16, "post", 1, 576, 24000, True), (torch.float32, "post", 2, 640, 24008, False),
    (torch.float32, "post", 2, 704, 24008, True), (torch.bfloat16, "mix2", 1, 704, 12008, False), (torch.bfloat16, "mix2", 1, 768, 12008, True), (torch.bfloat16, "mix2", 1, 704, 12000, True),
    (torch.float32, "mix2", 1, 576, 12008, True), (torch.bfloat16, "mix5", 8, 576, 2064, False), (torch.bfloat16, "mix5", 4, 768, 2064, True)])
def test_short_k_of_many_columns(dtype, kind, M, K, N, taken):
    x, gain = torch.randn(5, M, K, device=DEV), torch.ones(K, device=DEV)
    h, w, y = torch.empty(M, K, dtype=dtype, device=DEV), (torch.randn(N, K, device=DEV) * K ** -0.5).to(dtype), torch.full((M, N), 7.0, device=DEV)
    t, gate, n = torch.randn(M, K, device=DEV), torch.rand(M, K, device=DEV).to(dtype), int(kind[3:]) if kind[:3] == "mix" else 0
    src = dict(x=x, coef=gain[:5], n_terms=n) if n else dict(x=x[0], y=t, gate=gate, ldg=K, post_gain=gain)
    assert B.norm_linear(B.linear_args(h, w, y, M=M), None, gain, None, torch.empty(M, K, device=DEV), eps=1e-5, many=True, **src) == taken
    if not taken:
        assert bool((y == 7).all())
        return
    d = torch.float64
    row = x[:n].to(d).sum(0) if n else x[0].to(d) + rms(t.to(d) * gate.to(d), gain.to(d), 1e-5)
    want = rms(row, gain.to(d), 1e-5) @ w.to(d).T
    tol = 4e-6 * 5 * (1 + want.abs()) if dtype == torch.float32 else 6 * 2 ** -9 * 1.5 * (1 + want.abs())      # (as in test_norm_stream; sums are stored in fp32)
    assert bool(((y.to(d) - want).abs() <= tol).all())


@pytest.mark.parametrize("dtype,M,K,N", [(torch.bfloat16, 8, 2048, 5136), (torch.bfloat16, 3, 1024, 5136), (torch.float32, 8, 1024, 2048)])
def test_sums_are_those_of_the_products_launch(dtype, M, K, N):
    """Two runs of k, each summed over the waves, then one and the other: the bits of the products' own launch over the same normed rows (read out by weights of one)."""
    x, t = torch.randn(M, K, device=DEV), torch.randn(M, K, device=DEV)
    gate, gain = torch.rand(M, K, device=DEV).to(dtype), torch.randn(K, device=DEV)
    got = []
    for w in (torch.eye(K, device=DEV, dtype=dtype), (torch.randn(N, K, device=DEV) * K ** -0.5).to(dtype)):
        y = torch.full((M, w.shape[0]), float("nan"), device=DEV)
        assert B.norm_linear(B.linear_args(torch.empty(M, K, dtype=dtype, device=DEV), w, y, M=M), None, gain, None, torch.empty(M, K, device=DEV), eps=1e-5, x=x, y=t, gate=gate, ldg=K,
                             post_gain=gain, many=True)
        got.append(y)
    want = torch.empty(M, N, device=DEV)
    B.linear(got[0].to(dtype), w, want, M=M)
    assert torch.equal(got[1], want)


def test_what_it_does_not_take():
    """Sizes beyond its own, and results over the rows that are read: refused or not taken, and nothing done."""
    def ask(M, K, N, y=None, xo=None, act=torch.bfloat16):
        x, t = torch.randn(M, K, device=DEV), torch.randn(M, K, device=DEV)
        gate, gain = torch.rand(M, K, device=DEV).to(act), torch.ones(K, device=DEV)
        h, w = torch.empty(M, K, dtype=act, device=DEV), torch.randn(N, K, device=DEV).to(act)
        out = torch.full((M, N), 7.0, dtype=act, device=DEV) if y is None else x if y == "x" else t
        a = B.linear_args(h, w, out, M=M)
        before = out.clone()
        taken = B.norm_linear(a, None, gain, None, torch.empty(M, K, device=DEV) if xo is None else x, eps=1e-5, x=x, y=t, gate=gate, ldg=K, post_gain=gain, many=True)
        assert taken or torch.equal(out, before)
        return taken
    assert ask(8, 2048, 512) and ask(8, 1024, 512)
    assert not ask(9, 1024, 512) and not ask(8, 2112, 512) and not ask(8, 512, 512) and not ask(8, 1088, 512) and not ask(4, 1000, 64)
    assert not ask(4, 1024, 1024, y="x") and not ask(4, 1024, 1024, y="y")
    with pytest.raises(RuntimeError, match="pcb_norm_linear"):
        ask(4, 1024, 512, xo="x")
