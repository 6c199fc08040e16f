"""A long question over a long staged cache: slices of the staged keys and the keys of the question itself in one launch (pc_attn_wide.hip).  One to three row groups a
wave, several q-blocks, last ones of few rows, heads that fill the chip's CUs or not, a past length of the device.  Against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("H,Hkv,q_len,past", [(8, 8, 128, 1100), (8, 2, 129, 1024), (3, 3, 200, 2049), (40, 40, 259, 1500), (32, 32, 288, 1088), (5, 5, 289, 1300), (16, 4, 400, 1031)])
def test_staged_and_own_keys_in_one_launch(H, Hkv, q_len, past, monkeypatch):
    from promptcache_amd import _native as n
    monkeypatch.setenv("PC_ATTN_WIDE_MIN", "1024")
    D, kv, g = 128, past + q_len, torch.Generator(device=DEV).manual_seed(past + q_len)
    cap = kv + 3
    q32, k32, v32 = (torch.randn(s, generator=g, device=DEV) for s in ((q_len, H, D), (Hkv, kv, D), (Hkv, kv, D)))
    q, k, v = q32.half(), torch.full((Hkv, cap, D), float("nan"), device=DEV).half(), torch.full((Hkv, cap, D), float("nan"), device=DEV).half()
    ql = (q32 - q.float()).half()
    k[:, :kv], v[:, :kv] = k32.half(), v32.half()
    klo, vlo = ((t[:, past:] - t[:, past:].half().float()).half().contiguous() for t in (k32, v32))
    ws = torch.full((n.attn_workspace_bytes(1, H, D, q_len, kv) // 4,), float("nan"), device=DEV)
    oh = torch.full((1, q_len, H * D), float("nan"), device=DEV).half()
    ol = torch.full_like(oh, float("nan"))
    for dev_past in (None, torch.tensor([past], dtype=torch.int32, device=DEV)):
        n.attn_fwd(q, q_len * H * D, H * D, k, v, Hkv * cap * D, cap * D, oh, q_len * H * D, H * D, 1, H, Hkv, D, q_len, past, D ** -0.5, ws, q_lo=ql, out_lo=ol,
                   kv_lo=(klo, vlo, Hkv * q_len * D, q_len * D, -1), past_len_dev=dev_past)
        kf, vf = k[:, :kv].double(), v[:, :kv].double()
        kf[:, past:] += klo.double()
        vf[:, past:] += vlo.double()
        want = torch.empty((q_len, H, D), dtype=torch.float64, device=DEV)
        hidden = torch.arange(kv, device=DEV)[None, :] > past + torch.arange(q_len, device=DEV)[:, None]
        for h in range(H):
            s = ((q[:, h].double() + ql[:, h].double()) @ kf[h // (H // Hkv)].T * D ** -0.5).masked_fill(hidden, float("-inf"))
            want[:, h] = torch.softmax(s, -1) @ vf[h // (H // Hkv)]
        got = oh[0].double() + ol[0].double()
        # scores within a few 2^-24 of |q k| / sqrt(D) <= 8 and P in two pieces within 2^-22, of values of up to 5
        assert float((got - want.reshape(q_len, H * D)).abs().max()) <= 5 * 4 * (8 * 2.0 ** -24 + 2.0 ** -22)
