"""pcb_head_prep of heads that are whole 16-byte chunks against float64: heads of every lane count, one head and head counts that fill no wave, row counts
around a workgroup's share, turned ranges inside a head, gains, blends, kept rows, destinations by row offset (aligned or not), in place."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


def rnd(*shape, seed=0, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV, dtype)


def rel(got, want):
    return float((got.to(F64) - want).norm() / want.norm())


def turned(x, pos, freqs, mag, off, dims):
    """Neighbouring columns off .. off + dims of x [T, H, D]."""
    ang = pos.to(F64)[:, None] * freqs
    c, s = (torch.cos(ang) * mag)[:, None], (torch.sin(ang) * mag)[:, None]
    out = x.clone()
    a, b = x[..., off:off + dims:2], x[..., off + 1:off + dims:2]
    out[..., off:off + dims:2], out[..., off + 1:off + dims:2] = a * c - b * s, b * c + a * s
    return out


# fp32: a norm of up to 512 squares and five roundings; bf16 results half a last place
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-6), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("T", [1, 3, 64, 65, 1027])
@pytest.mark.parametrize("H,D,off,dims", [(5, 128, 0, 128), (16, 64, 16, 32), (1, 192, 0, 0), (1, 512, 128, 128), (3, 200, 8, 64), (9, 8, 0, 8), (2, 320, 0, 256)])
def test_heads_in_chunks(T, H, D, off, dims, dtype, tol):
    from promptcache_amd import _blocks as B
    G = 2
    N = (H + 2 * G) * D + 8
    P, gain, lam = rnd(T, N, seed=1, dtype=dtype), rnd(D, seed=2) + 1.0, torch.tensor([0.3], device=DEV)
    pos = torch.randperm(5000, generator=torch.Generator().manual_seed(3))[:T].to(DEV, torch.int32)
    freqs = torch.rand(max(dims // 2, 1), generator=torch.Generator().manual_seed(4), dtype=F64).to(DEV)[:dims // 2]
    cap = T + 3
    q, keep = torch.empty(T, H * D, dtype=dtype, device=DEV), torch.zeros(T, G * D, device=DEV)
    plane = torch.zeros(G, cap, 2 * D, dtype=dtype, device=DEV)
    rows = torch.randperm(cap, generator=torch.Generator().manual_seed(5))[:T].to(DEV)
    shift = 1 if D == 8 else 0                                   # (a cache that begins off the 16-byte grid: rows by element)
    off_rows = rows * 2 * D + shift
    other = rnd(T, G * D, seed=6)
    turn = dict(rot_dims=dims, rot_off=off) if dims else {}
    at = dict(row_off=off_rows, head_stride=cap * 2 * D)
    flat = torch.zeros(plane.numel() + 8, dtype=dtype, device=DEV)
    segs = [B.head_seg(P, N, H, D, q, norm=True, gain=gain, ld_dst=H * D, **turn),
            B.head_seg(P[:, H * D:], N, G, D, flat, norm=True, **turn, **at),
            B.head_seg(P[:, (H + G) * D:], N, G, D, flat, norm=True, blend=lam, other=other, keep=keep, dst_offset=D, **at)]
    kw = dict(eps=1e-6) if not dims else dict(eps=1e-6, pos=pos, freqs=freqs, rot_mag=1.1)
    B.head_prep(segs, T, dtype, **kw)
    x = P.to(F64)[:, :(H + 2 * G) * D].view(T, H + 2 * G, D)
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6)
    rot = (lambda v: turned(v, pos, freqs, 1.1, off, dims)) if dims else (lambda v: v)
    assert rel(q.view(T, H, D), rot(x[:, :H] * gain.to(F64))) < tol
    got = flat[shift:shift + plane.numel()].view(G, cap, 2 * D)[:, rows].transpose(0, 1)
    blended = 0.7 * x[:, H + G:] + 0.3 * other.to(F64).view(T, G, D)
    assert rel(got[..., :D], rot(x[:, H:H + G])) < tol and rel(got[..., D:], blended) < tol and rel(keep.view(T, G, D), blended) < 1e-6
    # in place, and the same turns from a table
    if dims:
        again = P.clone()
        table = torch.empty(T, dims, device=DEV)
        B.rot_table(pos, freqs, 1.1, table, T)
        B.head_prep([B.head_seg(again, N, H, D, again, norm=True, gain=gain, ld_dst=N, **turn)], T, dtype, eps=1e-6, table=table)
        assert torch.equal(again[:, :H * D], q) and torch.equal(again[:, H * D:], P[:, H * D:])


def test_a_head_that_is_no_number_stays_alone():
    from promptcache_amd import _blocks as B
    T, H, D = 70, 5, 64
    P = rnd(T, H * D, seed=1, dtype=torch.bfloat16)
    P[9, 2 * D + 3] = float("nan")
    q = torch.zeros_like(P)
    B.head_prep([B.head_seg(P, H * D, H, D, q, norm=True, ld_dst=H * D)], T, torch.bfloat16, eps=1e-6)
    bad = torch.isnan(q).view(T, H, D)
    assert bool(bad[9, 2].all()) and int(bad.sum()) == D
