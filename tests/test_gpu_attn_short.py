"""Attention of a few new rows over a staged cache at the edges of its dispatch: the pass's own rows on the matrix cores (one and two row tiles, every
head dim), fewer streams over short caches (768, 1024 keys), a row tile a workgroup or two in one, with and without ALiBi.  Against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _n():
    from promptcache_amd import _native
    return _native


@pytest.mark.parametrize("alibi", [False, True])
@pytest.mark.parametrize("H,Hkv,D,q_len,past", [
    (4, 2, 128, 1, 1), (4, 4, 64, 5, 40), (8, 8, 32, 16, 100), (4, 2, 128, 17, 3), (2, 2, 64, 32, 238), (32, 32, 128, 31, 60),       # the 64-row kernel beside the tail
    (32, 32, 128, 2, 254), (32, 32, 128, 3, 253), (8, 2, 128, 15, 768), (8, 2, 128, 16, 769), (40, 40, 128, 16, 1024), (40, 40, 128, 16, 1025),
    (32, 32, 128, 17, 239), (32, 32, 128, 27, 308), (8, 2, 64, 31, 768), (16, 16, 32, 32, 769), (40, 40, 128, 29, 700), (40, 40, 128, 32, 769),
    (54, 54, 128, 18, 300), (64, 64, 128, 20, 300), (32, 32, 128, 25, 1024), (32, 8, 128, 32, 1300),
    (40, 40, 128, 17, 1280), (40, 40, 128, 32, 1281), (40, 40, 64, 30, 1281)])                                     # (ALiBi, a wave's second tile: the 64-row kernel)
def test_a_few_rows_over_a_staged_cache(H, Hkv, D, q_len, past, alibi):
    n = _n()
    kv, g = past + q_len, torch.Generator().manual_seed(1000 * past + q_len)
    cap = kv + 5
    q32, k32, v32 = (torch.randn(s, generator=g) for s in ((q_len, H, D), (Hkv, kv, D), (Hkv, kv, D)))
    q, k, v = q32.half(), torch.full((Hkv, cap, D), float("nan")).half(), torch.full((Hkv, cap, D), float("nan")).half()
    ql = (q32 - q.float()).half()
    k[:, :kv], v[:, :kv] = k32.half(), v32.half()
    klo, vlo = ((t[:, past:] - t[:, past:].half().float()).half().contiguous() for t in (k32, v32))
    slopes = torch.exp2(-8.0 * torch.arange(1, H + 1) / H)
    kpos = torch.zeros(1, (kv + 63) // 64 * 64)
    kpos[0, :kv] = torch.arange(kv) * 2.0 - 2 * kv
    dev = [t.to(DEV) for t in (q, ql, k, v, klo, vlo, kpos, slopes * 1.4426950408889634)]
    ws = torch.full((max(n.attn_workspace_bytes(1, H, D, q_len, kv), 4) // 4,), float("nan"), dtype=torch.float32, device=DEV)
    mt = (q_len + 15) // 16
    oh = torch.full((mt, H * D // 32, 64, 8), float("nan"), dtype=torch.float16, device=DEV)
    ol = torch.full_like(oh, float("nan"))
    n.attn_fwd(dev[0], q_len * H * D, H * D, dev[2], dev[3], Hkv * cap * D, cap * D, None, 0, 0, 1, H, Hkv, D, q_len, past, D ** -0.5, ws, out_frag=(oh, ol), q_lo=dev[1],
               kv_lo=(dev[4], dev[5], Hkv * q_len * D, q_len * D, -1), alibi=(dev[6], dev[7]) if alibi else None)
    got = (n.from_act_frags(oh, q_len).double() + n.from_act_frags(ol, q_len).double()).cpu()
    kf, vf = k[:, :kv].double(), v[:, :kv].double()
    kf[:, past:] += klo.double()
    vf[:, past:] += vlo.double()
    kf, vf = (t.repeat_interleave(H // Hkv, 0) for t in (kf, vf))
    s = (q.double() + ql.double()).transpose(0, 1) @ kf.transpose(1, 2) * D ** -0.5
    bias = slopes.double()[:, None, None] * kpos.double()[:, None, :kv] if alibi else 0.0
    s = (s + bias).masked_fill(torch.arange(kv)[None, :] > past + torch.arange(q_len)[:, None], float("-inf"))
    want = (torch.softmax(s, -1) @ vf).transpose(0, 1).reshape(q_len, H * D)
    # a score is off by a few 2^-24 of the largest term of its sum (|q k| / sqrt(D) <= 8, a bias of up to 2 * 1332), P in two pieces by 2^-22 of itself, sums of
    # kv terms by sqrt(kv) 2^-24; each relative to values of up to 5: 4 (8 2^-24 + 2^-22) 5 without a bias, 2664 2^-24 5 more with one
    assert float((got - want).abs().max()) <= 5 * 4 * (8 * 2.0 ** -24 + 2.0 ** -22) + (5 * 2664 * 2.0 ** -24 if alibi else 0)


@pytest.mark.parametrize("H,Hkv,D,q_len,past", [(4, 4, 128, 3, 300), (8, 2, 64, 16, 40), (32, 32, 128, 16, 900), (4, 2, 128, 17, 300), (32, 32, 128, 27, 308), (40, 40, 128, 32, 40)])
@pytest.mark.parametrize("spread", [4.0, 12.0, 30.0, 45.0])
def test_a_large_value_on_an_unlikely_key_of_the_pass(H, Hkv, D, q_len, past, spread):
    """The weights of a pass's own keys are 32-bit numbers: a key of weight 2^-spread whose value is 2^14 times the others' counts with all of them."""
    n = _n()
    kv, g = past + q_len, torch.Generator().manual_seed(past + 7 * q_len)
    q32 = torch.zeros(q_len, H, D)
    q32[..., 0], q32[..., 1] = D ** 0.5, 0.3 * torch.randn(q_len, H, generator=g)
    k32, v32 = torch.zeros(Hkv, kv, D), torch.zeros(Hkv, kv, D)                      # (the staged keys: values of 0)
    k32[:, past:, 0] = -torch.rand(Hkv, q_len, generator=g)
    k32[:, past, 0] = -(spread + torch.rand(Hkv, generator=g)) * 0.6931471805599453
    k32[:, past:, 1] = torch.randn(Hkv, q_len, generator=g)
    k32[:, :past, 0] = -8.0
    v32[:, past:] = torch.randn(Hkv, q_len, D, generator=g)
    v32[:, past] *= 2.0 ** 12
    q, k, v = q32.half(), k32.half(), v32.half()
    ql = (q32 - q.float()).half()
    klo, vlo = ((t[:, past:] - t[:, past:].half().float()).half().contiguous() for t in (k32, v32))
    dev = [t.to(DEV) for t in (q, ql, k, v, klo, vlo)]
    ws = torch.full((max(n.attn_workspace_bytes(1, H, D, q_len, kv), 4) // 4,), float("nan"), dtype=torch.float32, device=DEV)
    mt = (q_len + 15) // 16
    oh = torch.full((mt, H * D // 32, 64, 8), float("nan"), dtype=torch.float16, device=DEV)
    ol = torch.full_like(oh, float("nan"))
    n.attn_fwd(dev[0], q_len * H * D, H * D, dev[2], dev[3], Hkv * kv * D, kv * D, None, 0, 0, 1, H, Hkv, D, q_len, past, D ** -0.5, ws, out_frag=(oh, ol), q_lo=dev[1],
               kv_lo=(dev[4], dev[5], Hkv * q_len * D, q_len * D, -1))
    got = (n.from_act_frags(oh, q_len).double() + n.from_act_frags(ol, q_len).double()).cpu()
    kf, vf = k.double(), v.double()
    kf[:, past:] += klo.double()
    vf[:, past:] += vlo.double()
    kf, vf = (t.repeat_interleave(H // Hkv, 0) for t in (kf, vf))
    s = (q.double() + ql.double()).transpose(0, 1) @ kf.transpose(1, 2) * D ** -0.5
    s = s.masked_fill(torch.arange(kv)[None, :] > past + torch.arange(q_len)[:, None], float("-inf"))
    p = torch.softmax(s, -1)
    want = (p @ vf).transpose(0, 1).reshape(q_len, H * D)
    # a term p v is off by what its score and the largest are (each a few 2^-24 of itself, up to 46 + 8 together) and some roundings of 2^-24 of products and sums;
    # the result, as two fp16 planes, by 2^-22 of itself and the smallest step of fp16
    terms = (p @ vf.abs()).transpose(0, 1).reshape(q_len, H * D)
    tol = terms * (4 * (spread + 8) + 8) * 2.0 ** -24 + 2.0 ** -22 * want.abs() + 2.0 ** -24
    assert float(((got - want).abs() / tol).max()) <= 1
