"""The row kernels that hold a row in registers (pcb_post_norm, pcb_mix_norm, pcb_polynorm) against float64: widths around the edges of a
thread's chunks and of the two ways to spread a row over threads (up to 512 rows, more than 512).

Tolerances: a sum of `width` fp32 squares in any order is off by at most width * 2^-24 of itself, in practice by its square root's share; 1e-6
leaves room for that at 16384 columns.  bf16 results (8 significant bits) add their own rounding, at most half a last place: 2^-8 of a value."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


def B():
    from promptcache_amd import _blocks
    return _blocks


def rnd(*shape, seed=0, scale=1.0, dtype=torch.float32):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(dtype)


def rel(got, want):
    got, want = got.to(F64), want.to(F64)
    return float((got - want).norm() / want.norm())


def unit(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("rows,width", [(3, 4), (1, 1020), (2, 1028), (5, 4100), (2, 16384), (2, 8190), (520, 1024), (520, 1032), (513, 4108)])
def test_rows_held_in_registers(rows, width, dtype, tol):
    eps, f = 1e-5, lambda t: t.to(F64)
    x0, y, add = rnd(rows, width, seed=1, scale=3.0), rnd(rows, width, seed=2), rnd(rows, width, seed=3)
    gate = rnd(rows, width + 4, seed=4).sigmoid().to(dtype)[:, 4:]
    pg, g, bias = 1 + 0.1 * rnd(width, seed=5), 1 + 0.1 * rnd(width, seed=6), rnd(width, seed=7)
    out, x_out = torch.empty(rows, width, dtype=dtype, device=DEV), torch.empty(rows, width, device=DEV)
    # both halves: gate, norm behind the sublayer, a second summand; then the layer norm of the result without them
    x = x0.clone()
    B().post_norm(x, y=y, gate=gate, ldg=width + 4, post_gain=pg, add=add, y_scale=0.7, gain=g, out=out, x_out=x_out, eps=eps)
    want = f(x0) + 0.7 * unit(f(y) * f(gate), eps) * f(pg) + f(add)
    assert rel(x, want) < 1e-6 and torch.equal(x, x_out) and rel(out, unit(want, eps) * f(g)) < tol
    B().post_norm(x, gain=g, bias=bias, layer_norm=True, out=out, eps=eps)
    d = f(x) - f(x).mean(-1, keepdim=True)
    assert rel(out, unit(d, eps) * f(g) + f(bias)) < tol
    # sums of streams, two norms
    for n in (1, 4, 5):
        hist, coef = rnd(n, rows, width, seed=8), rnd(n, seed=9)
        o2 = torch.empty_like(out)
        B().mix_norm(hist, n, coef, g, out, pg, o2, x_out=x_out, eps=eps, n_rows=rows)
        want = torch.einsum("n,nrw->rw", f(coef), f(hist))
        # (sums that cancel keep the rounding of their terms)
        assert rel(x_out, want) < 1e-6 and rel(out, unit(want, eps) * f(g)) < tol and rel(o2, unit(want, eps) * f(pg)) < tol
    # the polynomial of normed powers
    c = rnd(4, seed=10)
    B().polynorm(x0, c, out, eps, rows)
    z = f(x0)
    want = f(c)[0] * unit(z, eps) + f(c)[1] * unit(z ** 2, eps) + f(c)[2] * unit(z ** 3, eps) + f(c)[3]
    assert rel(out, want) < tol


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("rows,width", [(2, 4224), (2, 8192), (2, 8196), (2, 12288), (515, 3072), (513, 4100), (514, 5128), (513, 8192), (513, 8200)])
def test_rows_of_two_chunks_a_thread_and_wider(rows, width, dtype, tol):
    test_rows_held_in_registers(rows, width, dtype, tol)
