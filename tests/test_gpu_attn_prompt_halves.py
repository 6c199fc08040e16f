"""pcb_attn_prompt against float64 on both sides of its split of the key blocks: launches of few workgroups (two halves that share a tile's blocks, one of
them with none where a tile sees a single block) and of many (one)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


# weights carry 16 bits in bf16, results are rounded to 8; fp32: sums over up to 600 keys
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 3e-6), (torch.bfloat16, 4e-3)])
@pytest.mark.parametrize("dim,vdim", [(128, 128), (64, 64), (192, 128)])
@pytest.mark.parametrize("rows,H,block,window", [
    ([1, 63, 64, 65, 130], 4, 0, 0),            # few workgroups: tiles of one block, of two, of three
    ([600], 4, 256, 0),
    ([600], 4, 0, 70),
    ([600] * 3, 24, 256, 0),                    # 720 workgroups: one half
])
def test_both_sides_of_the_split(rows, H, block, window, dim, vdim, dtype, tol):
    from promptcache_amd import _blocks as B
    g = torch.Generator().manual_seed(len(rows))
    T, G = sum(rows), H // 2
    q, k, v = (torch.randn(T, n, generator=g).to(DEV, dtype) for n in (H * dim, G * dim, G * vdim))
    sink = torch.randn(H, generator=g).to(DEV)
    starts = [sum(rows[:b]) for b in range(len(rows))]
    tiles = torch.tensor([[s, at, min(64, n - at), s + at] for s, n in zip(starts, rows) for at in range(0, n, 64)], dtype=torch.int32, device=DEV)
    out = torch.full((T, H * vdim), float("nan"), device=DEV, dtype=dtype)
    B.attn_prompt(q, tiles.reshape(-1), tiles.shape[0], 64, k, (G * dim, dim), v, (G * vdim, vdim), H, G, dim, vdim, dim ** -0.5, out, ldo=H * vdim,
                  sink=sink, block=block, window=window)
    for s, n in zip(starts, rows):
        pos = torch.arange(n, device=DEV)
        dist = pos[:, None] - pos[None]
        hidden = dist < 0
        if block:
            hidden |= (pos // block)[:, None] != (pos // block)[None]
        if window:
            hidden |= dist >= window
        Q, K, V = q[s:s + n].to(F64).view(n, H, dim), k[s:s + n].to(F64).view(n, G, dim), v[s:s + n].to(F64).view(n, G, vdim)
        for h in range(H):
            w = (Q[:, h] @ K[:, h // 2].T * dim ** -0.5).masked_fill(hidden, float("-inf"))
            w = torch.softmax(torch.cat([w, sink[h].to(F64).expand(n, 1)], 1), -1)[:, :n]
            want, got = w @ V[:, h // 2], out[s:s + n, h * vdim:(h + 1) * vdim].to(F64)
            assert float((got - want).norm() / want.norm()) < tol, (s, h)


# (`longest` decides who shares a tile's blocks: what the launch is told of a longer context than there is changes its speed alone)
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 3e-6), (torch.bfloat16, 4e-3)])
@pytest.mark.parametrize("dim,vdim", [(128, 128), (64, 64), (192, 128), (100, 60)])
@pytest.mark.parametrize("rows,H,block,window", [([1, 63, 64, 65, 130], 4, 0, 0), ([600], 4, 512, 0), ([600], 4, 0, 300), ([600] * 3, 16, 0, 0), ([600] * 3, 24, 0, 0)])
def test_two_halves_of_a_tile(rows, H, block, window, dim, vdim, dtype, tol, monkeypatch):
    import functools
    from promptcache_amd import _blocks as B
    monkeypatch.setattr(B, "attn_prompt", functools.partial(B.attn_prompt, longest=2000))
    test_both_sides_of_the_split(rows, H, block, window, dim, vdim, dtype, tol)
