"""The decoding step of an attention layer in one launch behind its projection (pb_attn_step.hip), against torch in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
F64 = torch.float64


def B():
    from promptcache_amd import _blocks
    return _blocks


def rnd(*shape, seed, dtype=torch.float32, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(dtype).to(DEV)


def unit(x, eps):
    x = x.to(F64)
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def turned(x, pos, freqs, mag):
    """The first 2 x len(freqs) columns of x [rows, heads, columns], neighbouring pairs."""
    ang = pos.to(F64)[:, None] * freqs[None]
    c, s, n = torch.cos(ang)[:, None] * mag, torch.sin(ang)[:, None] * mag, 2 * freqs.numel()
    a, b = x[..., 0:n:2], x[..., 1:n:2]
    return torch.cat([torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2), x[..., n:]], -1)


def attended(q, keys, vals, pos, slot, scale, lo, sink):
    """q [rows, H, dim]; keys, vals [slots, H, cap, columns] in 64 bits; one row's keys lo[r] .. pos[r]."""
    out = []
    for r in range(q.shape[0]):
        k, v = keys[slot[r], :, lo[r]:pos[r] + 1], vals[slot[r], :, lo[r]:pos[r] + 1]
        s = (k @ q[r][..., None])[..., 0] * scale
        if sink is not None:
            s = torch.cat([s, sink[:, None]], 1)
        p = torch.softmax(s, -1)[:, :k.shape[1]]
        out.append((p[:, None] @ v)[:, 0])
    return torch.stack(out)


# positions on both sides of the kernels' blocks of 32 and 64 keys, the first token of all, contexts in runs that some rows leave empty
POS = [0, 1, 31, 32, 63, 64, 65, 127, 200, 299]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,G,D,Dv,rot,block,window", [(16, 4, 128, 128, 128, 0, 0), (8, 2, 64, 64, 32, 128, 0), (34, 2, 72, 40, 64, 0, 48), (4, 4, 128, 24, 0, 0, 0),
                                                       (3, 1, 8, 128, 8, 64, 100)])
@pytest.mark.parametrize("splits", [1, 3, 11])
def test_heads(dtype, H, G, D, Dv, rot, block, window, splits):
    b, n, cap, eps = B(), len(POS), 304, 1e-6
    HD, GD, GV = H * D, G * D, G * Dv
    pad = -(HD + GD + GV + H) % 8 + (1 if block else 0)          # (rows of whole 16 bytes, and others)
    P = rnd(n, HD + GD + GV + H + pad, seed=1, dtype=dtype)
    plane = rnd(n + 2, G, cap, D + Dv, seed=2, dtype=dtype)
    plane[:, :, :] = torch.where(torch.arange(cap, device=DEV)[:, None] < 300, plane, torch.full_like(plane, float("nan")))
    slot = [(5 * i + 1) % (n + 2) for i in range(n)]
    for r, p in enumerate(POS):
        plane[slot[r], :, p:] = float("nan")                     # (what is not written yet may hold anything)
    before = plane.clone()
    rows = torch.randperm(n, generator=torch.Generator().manual_seed(3)).tolist()
    tiles = torch.tensor([[slot[r], POS[r], 1, r] for r in rows], dtype=torch.int32, device=DEV).reshape(-1)
    qg, kg, sink, lam, other = rnd(D, seed=4), rnd(D, seed=5), rnd(H, seed=6), torch.tensor([0.35], device=DEV), rnd(n, GV, seed=7)
    freqs = torch.tensor([1000.0 ** (-2 * i / max(rot, 1)) for i in range(rot // 2)], dtype=F64, device=DEV)
    keep, out = torch.zeros(n, GV, device=DEV), torch.zeros(n, H * Dv, dtype=dtype, device=DEV)
    part = torch.full((b.attn_softmax_part(n, H, splits, Dv),), float("nan"), device=DEV) if splits > 1 else None
    strides = (G * cap * (D + Dv), cap * (D + Dv), D + Dv)
    assert b.attn_step_fits(dtype, H, G, D, Dv, rot)
    kw = dict(q_at=0, q_head_stride=D, k_at=HD, v_at=HD + GD, q_gain=qg, k_gain=kg, eps=eps, rot_dims=rot, freqs=freqs if rot else None, rot_mag=1.25, blend=lam,
              other=other, keep=keep, window=window, block=block, sink=sink, gate=P[:, HD + GD + GV:], ldg=P.shape[1])
    b.attn_step(P, tiles, n, plane, strides, plane.view(-1)[D:], strides, H, G, D, Dv, D ** -0.5, out, n_splits=splits, part=part, **kw)
    pos = torch.tensor(POS, device=DEV)
    q = turned(unit(P[:, :HD].view(n, H, D), eps) * qg.to(F64), pos, freqs, 1.25)
    k = turned(unit(P[:, HD:HD + GD].view(n, G, D), eps) * kg.to(F64), pos, freqs, 1.25)
    v0 = unit(P[:, HD + GD:HD + GD + GV].view(n, G, Dv), eps)
    v = (1 - lam.to(F64)) * v0 + lam.to(F64) * other.to(F64).view(n, G, Dv)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -21   # (a value computed in fp32 and stored: half a step of bf16, or a few of fp32; 2^-19: of the pair that is turned)
    assert float((keep.view(n, G, Dv).to(F64) - v).abs().max()) <= 2.0 ** -21 * float(v.abs().max())
    new = torch.stack([plane[slot[r], :, POS[r]] for r in range(n)]).to(F64)
    assert bool(((new - torch.cat([k, v], -1)).abs() <= ulp * torch.cat([k, v], -1).abs() + 2.0 ** -19).all())
    for r in range(n):                                           # nothing else was written
        plane[slot[r], :, POS[r]] = before[slot[r], :, POS[r]]
    assert torch.equal(plane.view(torch.int16 if dtype == torch.bfloat16 else torch.int32), before.view(torch.int16 if dtype == torch.bfloat16 else torch.int32))
    full = before.to(F64)
    for r in range(n):
        full[slot[r], :, POS[r]] = new[r]
    lo = [max(p - window + 1 if window else 0, p // block * block if block else 0, 0) for p in POS]
    want = attended(q.to(dtype).to(F64), full[..., :D].repeat_interleave(H // G, 1), full[..., D:].repeat_interleave(H // G, 1), POS, slot, D ** -0.5, lo, sink.to(F64))
    want = want * P[:, HD + GD + GV:HD + GD + GV + H].to(F64)[..., None]
    got = out.view(n, H, Dv).to(F64)
    # (bf16: the result's rounding, and queries that round the other way where fp32 and 64 bits fall on either side of a tie)
    tol = 6e-3 if dtype == torch.bfloat16 else 4e-6
    assert float((got - want).norm() / want.norm()) < tol, float((got - want).norm() / want.norm())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("H,C,R,window", [(16, 192, 64, 0), (20, 64, 32, 100), (3, 32, 8, 0), (2, 160, 0, 33)])
@pytest.mark.parametrize("splits,up", [(1, 0), (4, 0), (1, 72), (4, 128), (11, 8), (64, 120)])
def test_latent(dtype, H, C, R, window, splits, up):
    """``up``: the heads' up-projections and gates in the merging launch."""
    b, n, cap, eps, D = B(), len(POS), 304, 1e-6, 24
    CR, DR, HQ = C + R, D + R, H * (D + R)
    P = rnd(n, HQ + CR + 8, seed=1, dtype=dtype)
    qa = rnd(n, H * CR, seed=2, dtype=dtype, scale=0.5)
    plane = rnd(n + 1, cap, CR, seed=3, dtype=dtype)
    slot = [(4 * i + 2) % (n + 1) for i in range(n)]
    for r, p in enumerate(POS):
        plane[slot[r], p:] = float("nan")
    before = plane.clone()
    tiles = torch.tensor([[slot[r], POS[r], 1, r] for r in range(n)], dtype=torch.int32, device=DEV).reshape(-1)
    gain, out = rnd(C, seed=4), torch.zeros(n, H * C, dtype=dtype, device=DEV)
    freqs = torch.tensor([100.0 ** (-2 * i / max(R, 1)) for i in range(R // 2)], dtype=F64, device=DEV)
    part = torch.full((b.attn_softmax_part(n, H, splits, C),), float("nan"), device=DEV) if splits > 1 or up else None
    kw = {}
    if up:
        w, gate, out = rnd(H, up, C, seed=5, dtype=dtype, scale=C ** -0.5), rnd(n, H * up + 8, seed=6, dtype=dtype), torch.zeros(n, H * up, dtype=dtype, device=DEV)
        kw = dict(up=w, up_gate=gate[:, 3:], ld_up_gate=H * up + 8)
    assert b.attn_step_fits(dtype, H, 1, CR, C, R, True)
    scale = 0.5 * CR ** -0.5
    b.attn_step(P, tiles, n, plane, (cap * CR, 0, CR), plane, (cap * CR, 0, CR), H, 1, CR, C, scale, out, q_at=D, q_head_stride=DR, k_at=HQ, q=qa, k_gain=gain,
                eps=eps, rot_dims=R, freqs=freqs if R else None, rot_mag=0.75, window=window, n_splits=splits, part=part, **kw)
    pos = torch.tensor(POS, device=DEV)
    c = unit(P[:, HQ:HQ + C], eps) * gain.to(F64)
    k = torch.cat([c, turned(P[:, None, HQ + C:HQ + CR].to(F64), pos, freqs, 0.75)[:, 0]], -1)
    q = torch.cat([qa.view(n, H, CR)[..., :C].to(F64), turned(P[:, :HQ].view(n, H, DR)[..., D:].to(F64), pos, freqs, 0.75)], -1)
    ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -21
    new = torch.stack([plane[slot[r], POS[r]] for r in range(n)]).to(F64)
    assert bool(((new - k).abs() <= ulp * k.abs() + 2.0 ** -19).all())
    full = before.to(F64)
    for r in range(n):
        full[slot[r], POS[r]] = new[r]
    full = full[:, None].expand(-1, H, -1, -1)
    want = attended(q.to(dtype).to(F64), full, full[..., :C], POS, slot, scale, [max(0, p - window + 1) if window else 0 for p in POS], None)
    if up:
        want = (w.to(F64) @ want[..., None])[..., 0] * gate[:, 3:3 + H * up].to(F64).view(n, H, up)
    got = out.view(n, H, up or C).to(F64)
    assert float((got - want).norm() / want.norm()) < (6e-3 if dtype == torch.bfloat16 else 4e-6)


def test_what_is_refused():
    b = B()
    for sizes in ((8, 2, 136, 128, 64), (8, 2, 128, 136, 64), (8, 2, 60, 64, 0), (8, 2, 64, 64, 4), (9, 2, 64, 64, 0), (8, 2, 32, 64, 64)):
        assert not b.attn_step_fits(torch.bfloat16, *sizes)
    for sizes in ((16, 1, 272, 208, 64), (16, 1, 256, 192, 32), (16, 2, 256, 192, 64), (16, 1, 240, 176, 64), (16, 1, 264, 192, 72)):
        assert not b.attn_step_fits(torch.float32, *sizes, True)
    P, plane, out = torch.zeros(1, 300, dtype=torch.bfloat16, device=DEV), torch.zeros(1, 1, 4, 132, dtype=torch.bfloat16, device=DEV), torch.zeros(1, 64, dtype=torch.bfloat16, device=DEV)
    tiles = torch.zeros(4, dtype=torch.int32, device=DEV)
    for dim, row, why in ((64, 132, "whole 16 bytes"), (60, 128, "does not take")):     # (cached rows of 132 elements)
        with pytest.raises(RuntimeError, match=why):
            b.attn_step(P, tiles, 1, plane, (4 * row, 4 * row, row), plane.view(-1)[64:], (4 * row, 4 * row, row), 1, 1, dim, 64, 1.0, out, q_at=0, q_head_stride=64, k_at=64,
                        v_at=128, eps=1e-6)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("splits", [0, -3])
def test_fewer_than_one_run_is_one(dtype, splits):
    """With the up-projections in the merging launch: what the first launch leaves is found by the second."""
    import ctypes
    b, n, H, C, R, up = B(), 3, 4, 64, 16, 24
    CR, HQ = C + R, H * (8 + R)
    P, qa, w, gate = rnd(n, HQ + CR, seed=1, dtype=dtype), rnd(n, H * CR, seed=2, dtype=dtype), rnd(H, up, C, seed=3, dtype=dtype), rnd(n, H * up, seed=4, dtype=dtype)
    plane, freqs = rnd(n, 40, CR, seed=5, dtype=dtype), torch.tensor([0.5 ** i for i in range(R // 2)], dtype=F64, device=DEV)
    tiles = torch.tensor([[r, 13 * r + 2, 1, r] for r in range(n)], dtype=torch.int32, device=DEV).reshape(-1)
    lib, got = b.load(), []
    real = lib.pcb_attn_step
    for s in (1, splits):
        part, out = torch.full((b.attn_softmax_part(n, H, 1, C),), float("nan"), device=DEV), torch.zeros(n, H * up, dtype=dtype, device=DEV)

        def call(args, stream):                                  # (the wrapper counts such runs as one itself)
            args._obj.n_splits = s
            return real(ctypes.byref(args._obj), stream)
        try:
            lib.pcb_attn_step = call
            b.attn_step(P, tiles, n, plane, (40 * CR, 0, CR), plane, (40 * CR, 0, CR), H, 1, CR, C, 0.1, out, q_at=8, q_head_stride=8 + R, k_at=HQ, q=qa, eps=1e-6,
                        rot_dims=R, freqs=freqs, part=part, up=w, up_gate=gate, ld_up_gate=H * up, n_splits=s)
        finally:
            lib.pcb_attn_step = real
        got.append(out)
    assert bool(torch.isfinite(got[0]).all()) and torch.equal(got[0], got[1])
