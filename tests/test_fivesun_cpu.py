"""CPU-side checks of the Fivesun integration: configuration reader, tensor naming, checkpoint directories, the arena's planes and
states for this design, the blocks library's new argument structures, the frequency tables the model hands to its kernels, and
properties of the plain oracle itself (each mechanism made visible by inputs built for it)."""
import ctypes
import json
import math
import os
import subprocess

import pytest
import torch

from oracle import fivesun_oracle as O
from promptcache_amd.model import weights as W
from promptcache_amd.model.config import FivesunLayer, FivesunShape, architecture_of

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F = torch.float64


def small_shape():
    return FivesunShape(vocab_size=60, hidden_size=24, norm_eps=1e-5, embed_scale=3.5, layers=[
        FivesunLayer("mlstm", heads=2, kv_heads=2, dim=6, vdim=8, gate_cap=4.0, ff=16),
        FivesunLayer("attention", heads=4, kv_heads=2, dim=8, vdim=6, scale=0.3, mask=5, rot_base=100.0, rot_dims=4, rot_factor=2.0, v_mix=True),
        FivesunLayer("latent_attention", heads=3, kv_heads=1, dim=6, vdim=4, kv_rank=10, rot_dim=4, rot_dims=4, scale=0.25, mask=4,
                     rot_base=50.0, rot_factor=4.0, yarn_original=16.0, yarn_fast=4.0, yarn_slow=1.0, ff=12),
        FivesunLayer("attention", heads=2, kv_heads=2, dim=8, vdim=6, scale=0.4, mask=0, rot_base=100.0, rot_dims=8, rot_factor=1.0, v_mix=True, ff=8),
    ])


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=F)


# ---- configuration and tensors -------------------------------------------------------------------------------------------------
def test_config_round_trip_and_every_branch(tmp_path):
    s = small_shape()
    c = s.to_config()
    assert c["architecture"] == "Fivesun" and c["layers"][1]["mlp"] is None and c["layers"][3]["mixer"].get("mask") is None
    assert c["layers"][2]["mixer"]["rot"]["scaling"]["original"] == 16.0 and c["embedding"]["scale"] == 3.5
    back = FivesunShape.from_config(json.loads(json.dumps(c)))
    assert back.to_config() == c and back.first_v_mix == 1 and [l.kind for l in back.layers] == [l.kind for l in s.layers]
    (tmp_path / "config.json").write_text(json.dumps(c))
    assert architecture_of(str(tmp_path)) == "fivesun"
    # what a configuration leaves out does not exist: no mask, no scaling, key heads = query heads, value size = key size
    lean = {"architecture": "Fivesun", "vocab": 9, "width": 8, "layers": [
        {"type": "attention", "mixer": {"heads": 2, "dim": 4, "rot": {"base": 10.0, "dims": 2}}, "mlp": None}]}
    l = FivesunShape.from_config(lean).layers[0]
    assert (l.kv_heads, l.vdim, l.mask, l.rot_factor, l.v_mix, l.ff, l.rot_dims) == (2, 4, 0, 1.0, False, 0, 2)
    for bad in ({"type": "conv"}, {"type": "attention", "mixer": {"heads": 3, "kv_heads": 2, "dim": 4}},
                {"type": "attention", "mixer": {"heads": 2, "dim": 4, "rot": {"dims": 3}}},
                {"type": "latent_attention", "mixer": {"heads": 2, "dim": 4, "kv_rank": 4, "rot_dim": 2, "rot": {"dims": 4}}},
                {"type": "mlstm", "mixer": {"heads": 2, "dim": 4}, "mlp": {"kind": "moe", "ff": 4}}):
        with pytest.raises(ValueError):
            FivesunShape.from_config(dict(lean, layers=[bad]))
    # blended values must have the first blending layer's shape
    two = [{"type": "attention", "mixer": {"heads": 2, "dim": 4, "v_mix": True}}, {"type": "attention", "mixer": {"heads": 2, "dim": 4, "vdim": 6, "v_mix": True}}]
    with pytest.raises(ValueError):
        FivesunShape.from_config(dict(lean, layers=two))


def test_tensor_names_and_checkpoint_directory(tmp_path):
    from safetensors.torch import save_file
    s = small_shape()
    shapes = W.fivesun_weight_shapes(s)
    assert shapes["l1.mix.sink"] == (4,) and shapes["l1.mix.g"] == (4, 24) and shapes["l1.mix.vmix"] == () and "l1.norm2" not in shapes
    assert shapes["l2.mix.dkv"] == (14, 24) and shapes["l2.mix.uk"] == (18, 10) and shapes["l2.mix.q"] == (30, 24)
    assert shapes["l0.mix.i"] == (2, 24) and shapes["l0.mix.norm"] == (16,) and shapes["l0.mlp.down.b"] == (24,) and shapes["l0.rg2"] == (24, 24)
    w = W.make_fivesun_weights(s, seed=2)
    assert set(w) == set(shapes) and all(tuple(w[k].shape) == tuple(v) and w[k].dtype == torch.bfloat16 for k, v in shapes.items())
    assert 0.0 < float(w["l3.mix.vmix"]) < 1.0 and float(w["l1.mix.sink"].float().abs().min()) > 0.0
    (tmp_path / "config.json").write_text(json.dumps(s.to_config()))
    save_file({k: v.contiguous() for k, v in w.items()}, str(tmp_path / "model.safetensors"))
    back = W.load_fivesun_safetensors(str(tmp_path), FivesunShape.from_dir(str(tmp_path)))
    assert all(torch.equal(back[k], w[k]) for k in w)
    w2 = dict(w)
    w2["l2.mix.uv"] = w["l2.mix.uv"][:, :-1].contiguous()
    save_file({k: v.contiguous() for k, v in w2.items()}, str(tmp_path / "model.safetensors"))
    with pytest.raises(ValueError):
        W.load_fivesun_safetensors(str(tmp_path), s)
    del w2["l2.mix.uv"]
    save_file({k: v.contiguous() for k, v in w2.items()}, str(tmp_path / "model.safetensors"))
    with pytest.raises(KeyError):
        W.load_fivesun_safetensors(str(tmp_path), s)


def test_arena_serial_numbers_never_repeat():
    from promptcache_amd.model.kv_arena import SlotArena
    seen = set()
    for _ in range(5):
        ar = SlotArena([(1, 4)], 1, 4, "cpu", torch.float32)
        assert ar.serial not in seen
        seen.add(ar.serial)
        del ar


def step_tables(m, arena, slots, tokens):
    """The tables a step of model ``m`` hands its launches, as lists (nothing is launched), and what its block is made of."""
    seen = []
    m._run = lambda arena, blob, dims, logits, *_: seen.append((m._tables(blob, dims), dims)) or logits
    m._decode_graphed = lambda arena, blob, dims: m._run(arena, torch.from_numpy(blob), dims, torch.zeros(dims["T"], m.V))
    m.forward_rows(arena, slots, tokens)
    (tb, dims), = seen
    return {k: v.tolist() if torch.is_tensor(v) else v for k, v in tb.items()}, dims


@pytest.mark.parametrize("prompt_rows", [16, 1])
@pytest.mark.parametrize("route", ["all", "tiled", "rebuilt", "last", "none", "rule"])
@pytest.mark.parametrize("news", [[1], [1, 1, 1], [16], [2, 15, 3], [17, 1, 40], [1, 200, 16, 3], [16, 64, 130]])
def test_step_tables_name_every_row_once(news, route, prompt_rows):
    """Which launch of a step takes which row, in plain words, whatever requests of 16 new tokens and more attend in tiles and whichever have their
    keys rebuilt -- and single rows only in a step that may be captured, whatever the knobs say."""
    from promptcache_amd.model.fivesun_hip import FivesunHIP
    lat = dict(heads=2, kv_heads=1, kv_rank=24, rot_dim=8, rot_dims=8, vdim=16)
    s = FivesunShape(vocab_size=50, hidden_size=32, norm_eps=1e-6, layers=[
        FivesunLayer("attention", heads=2, kv_heads=1, dim=16, vdim=16, mask=64, rot_dims=16), FivesunLayer("latent_attention", dim=16, mask=600, **lat),
        FivesunLayer("latent_attention", dim=256, mask=80, **lat), FivesunLayer("attention", heads=1, kv_heads=1, dim=264, vdim=8, rot_dims=0)])
    m = FivesunHIP(s, W.make_fivesun_weights(s, seed=1), device="cpu", dtype=torch.float32)
    m.PROMPT_ROWS, rule = prompt_rows, m._tiled
    pick = dict(all=lambda layers, cand, *_: list(cand), none=lambda *_: [], tiled=lambda layers, cand, *_: list(cand) if layers is m._att else [],
                rebuilt=lambda layers, cand, *_: list(cand) if layers is m._lat else [], last=lambda layers, cand, *_: cand[-1:], rule=rule)[route]
    m._tiled = lambda *a: picked.setdefault("att" if a[0] is m._att else "lat", pick(*a))
    picked = {}
    cap, starts = 4096, [1700, 0, 333, 70][:len(news)]
    ar = m.new_arena(5, cap)
    slots = [ar.alloc() for _ in range(5)][5 - len(news):]
    for b, n in enumerate(starts):
        ar.lengths[slots[b]] = n
    tb, dims = step_tables(m, ar, slots, [[7] * n for n in news])
    T, flat = sum(news), [sum(news[:b]) for b in range(len(news))]
    row = {flat[b] + i: [slots[b], starts[b] + i, 1, flat[b] + i] for b in range(len(news)) for i in range(news[b])}
    one = all(n == 1 for n in news)
    big, rebuilt = picked["att"], picked["lat"]
    assert all(news[b] >= prompt_rows and not one for b in big + rebuilt)
    low = {b: max(0, starts[b] - 599) // 64 * 64 for b in rebuilt}
    single = [r for b in range(len(news)) if b not in big for r in range(flat[b], flat[b] + news[b])]
    folded = [r for b in range(len(news)) if b not in rebuilt for r in range(flat[b], flat[b] + news[b])]

    def quads(t):
        return [t[i:i + 4] for i in range(0, len(t), 4)]
    assert [tb["pos"][r] for r in range(T)] == [row[r][1] for r in range(T)] and len(tb["ids"]) == T
    assert quads(tb["s_tiles"]) == [row[r] for r in single] and quads(tb["f_tiles"]) == [row[r] for r in folded]
    assert tb["f_rows"] == (folded if rebuilt else []) and quads(tb["a_tiles"]) == ([row[r] for r in range(T)] if rebuilt else [])
    assert sorted(quads(tb["w_tiles"])) == sorted([slots[b], starts[b] + q, min(16, news[b] - q), flat[b] + q] for b in range(len(news)) for q in range(0, news[b], 16))
    # tiles: every row of theirs once, its own request's; rebuilt rows hold what the window can see of it
    for tiles, which in ((quads(tb["p_tiles"]), big), (quads(tb["l_tiles"]), rebuilt)):
        got = sorted(r for t in tiles for r in range(t[3], t[3] + t[2]))
        assert got == [r for b in which for r in range(flat[b], flat[b] + news[b])] and all(0 < t[2] <= tb["tile"] for t in tiles)
        assert all(row[t[3]][1] == t[1] for t in tiles)
    assert all(t[0] == row[t[3]][0] for t in quads(tb["p_tiles"]))
    for base, p0, n, r in quads(tb["l_tiles"]):
        b = next(b for b in rebuilt if flat[b] <= r < flat[b] + news[b])
        assert [tb["kv_rows"][base + j] for j in range(low[b], p0 + n)] == [slots[b] * cap + j for j in range(low[b], p0 + n)]
    assert [x for x in tb["offs"]] == [[row[r][0] * g * cap * d + row[r][1] * d for r in range(T)] for g, d in m._sigs]
    if one:                                        # launches of a captured step do not depend on how long its requests are
        for b in range(len(news)):
            ar.lengths[slots[b]] = 5 + b
        assert step_tables(m, ar, slots, [[7] * n for n in news])[1] == dims


def test_long_contexts_with_few_new_tokens_are_not_tiled():
    """The measured sides of the rule: a lone portion over a long context goes row by row, a prompt in tiles, many portions together in tiles,
    and a portion over a long context does not hold up the prompt beside it (16 heads over 4, a latent of 192)."""
    from promptcache_amd.model.fivesun_hip import FivesunHIP
    lat = dict(heads=16, kv_heads=1, kv_rank=192, rot_dim=64, rot_dims=64, dim=128, vdim=128)
    s = FivesunShape(vocab_size=50, hidden_size=32, norm_eps=1e-6, layers=[
        FivesunLayer("attention", heads=16, kv_heads=4, dim=128, vdim=128, rot_dims=128), FivesunLayer("latent_attention", **lat)])
    m = FivesunHIP(s, W.make_fivesun_weights(s, seed=1), device="cpu", dtype=torch.bfloat16)
    for news, starts, att, latent in [([16], [30000], [], []), ([64], [8000], [], []), ([256], [30000], [0], []), ([2048], [0], [0], [0]),
                                      ([64] * 8, [8000] * 8, list(range(8)), []), ([256] * 8, [8000] * 8, list(range(8)), list(range(8))),
                                      ([300] * 8, [0] * 8, list(range(8)), list(range(8))), ([16, 2048], [30000, 0], [1], [1])]:
        cand = list(range(len(news)))
        assert m._tiled(m._att, cand, news, starts) == att and m._tiled(m._lat, cand, news, starts) == latent, (news, starts)


def test_frequency_tables_follow_the_oracle():
    from promptcache_amd.model.fivesun_hip import rotary_frequencies
    fr, mag = rotary_frequencies(30000.0, 12, 3.0)
    want, wm = O.plain_frequencies(30000.0, 12, 3.0)
    assert mag == wm == 1.0 and torch.allclose(torch.from_numpy(fr), want, rtol=1e-14)
    for args in ((70000.0, 32, 3.0, 1024.0, 16.0, 2.0), (10000.0, 8, 4.0, 64.0, 8.0, 1.0), (100.0, 4, 8.0, 16.0, 2.0, 0.5)):
        fr, mag = rotary_frequencies(*args)
        want, wm = O.yarn_frequencies(*args)
        assert abs(mag - wm) < 1e-15 and torch.allclose(torch.from_numpy(fr), want, rtol=1e-14)


# ---- the blocks library's argument structures --------------------------------------------------------------------------------------
def test_blocks_struct_layouts_match_the_header(tmp_path):
    from promptcache_amd import _blocks
    structs = (("pcb_post_norm_args", _blocks.PostNormArgs), ("pcb_head_prep_seg", _blocks.HeadPrepSeg), ("pcb_head_prep_args", _blocks.HeadPrepArgs),
               ("pcb_mlstm_args", _blocks.MlstmArgs), ("pcb_attn_softmax_args", _blocks.AttnSoftmaxArgs), ("pcb_linear_args", _blocks.LinearArgs))
    body = ['#include <stdio.h>', '#include <stddef.h>', f'#include "{ROOT}/include/promptcache_blocks.h"', 'int main(void) {']
    for st, cls in structs:
        body.append(f'  printf("{st} %zu\\n", sizeof({st}));')
        for f, _ in cls._fields_:
            body.append(f'  printf("{st}.{f} %zu\\n", offsetof({st}, {f}));')
    body += ['  return 0;', '}']
    src = tmp_path / "layout.c"
    src.write_text("\n".join(body))
    exe = tmp_path / "layout"
    subprocess.check_call(["gcc", "-std=c99", "-Wall", "-Werror", str(src), "-o", str(exe)])
    got = dict(line.rsplit(" ", 1) for line in subprocess.check_output([str(exe)], text=True).strip().splitlines())
    for st, cls in structs:
        assert int(got[st]) == ctypes.sizeof(cls), st
        for name, _ in cls._fields_:
            assert int(got[f"{st}.{name}"]) == getattr(cls, name).offset, (st, name)


def test_blocks_reject_bad_arguments_on_the_host():
    from promptcache_amd import _blocks
    assert os.path.exists(_blocks.lib_path()), "run __graft_entry__.build() first"
    lb = _blocks.load(build_missing=False)
    a = _blocks.PostNormArgs(ctypes.sizeof(_blocks.PostNormArgs), 0, None, None, None, 0, None, None, None, None, None, 1e-6, 2, 20000)
    assert lb.pcb_post_norm(ctypes.byref(a), None) == -2001 and b"width" in lb.pcb_last_error_string()
    a.width = 8
    assert lb.pcb_post_norm(ctypes.byref(a), None) == -2001 and b"null pointer" in lb.pcb_last_error_string()
    a.struct_bytes -= 4
    assert lb.pcb_post_norm(ctypes.byref(a), None) == -2001 and b"struct size" in lb.pcb_last_error_string()
    m = _blocks.MlstmArgs(ctypes.sizeof(_blocks.MlstmArgs), 0, None, None, None, None, None, 600, 600, 16, 2, 2, None, 1, None, 10 ** 6, 2, 300, 8,
                          1.0, 0.0, None, 16)
    assert lb.pcb_mlstm(ctypes.byref(m), None) == -2001 and b"256 key columns" in lb.pcb_last_error_string()
    h = _blocks.HeadPrepArgs(ctypes.sizeof(_blocks.HeadPrepArgs), 0, 0, 1, None, None, 1.0, 1e-6)
    h.seg[0] = _blocks.HeadPrepSeg(None, 8, 8, 1, 8, 0, None, None, None, 0, None, 0, 3, 4, None, 8, None, 8, 1)
    assert lb.pcb_head_prep(ctypes.byref(h), None) == -2001 and b"pairs" in lb.pcb_last_error_string()      # an odd first rotated column
    assert lb.pcb_gated_norm(None, 12, None, None, 0, None, 12, 0, 1e-6, 2, 12, 5, 0, None, 0, None, 0, None) == -2001 and b"divide" in lb.pcb_last_error_string()
    assert lb.pcb_embed_scaled_rows(None, 0, None, 2.0, None, 3, 8, 10, None) == -2001 and b"null pointer" in lb.pcb_last_error_string()


# ---- the oracle's own properties ---------------------------------------------------------------------------------------------------
def test_oracle_forward_does_not_look_ahead_carries_its_state_and_layers_matter():
    s = small_shape()
    p = O.to_f64(W.make_fivesun_weights(s, seed=5))
    t = torch.randint(0, s.vocab_size, (19,), generator=torch.Generator().manual_seed(1)).tolist()
    full, streams, _ = O.forward(s, p, t)
    assert torch.allclose(O.forward(s, p, t[:9])[0], full[:9], atol=1e-10) and streams.shape == (4, 19, 24)
    a, _, carry = O.forward(s, p, t[:11])
    b, _, carry = O.forward(s, p, t[11:12], pos0=11, carry=carry)
    c, _, _ = O.forward(s, p, t[12:], pos0=12, carry=carry)
    assert torch.allclose(torch.cat([a, b, c]), full, atol=1e-9)
    for i in range(1, 4):
        assert float((streams[i] - streams[i - 1]).abs().max()) > 1e-3
    # the blend reaches layer 3 from layer 1: another blend weight changes the result, and so do layer 1's own values
    p2 = dict(p)
    p2["l3.mix.vmix"] = p["l3.mix.vmix"] + 0.2
    assert float((O.forward(s, p2, t)[0] - full).abs().max()) > 1e-4
    p2 = dict(p)
    p2["l1.mix.vmix"] = p["l1.mix.vmix"] + 0.2              # (the first blending layer's own weight is not used)
    assert torch.equal(O.forward(s, p2, t)[0], full)


def test_oracle_rotation_depends_on_distance_only_and_leaves_the_rest():
    fr, mag = O.plain_frequencies(100.0, 4, 2.0)
    assert torch.allclose(fr, torch.tensor([0.5, 0.05], dtype=F))
    q, k = rnd(1, 6, seed=1), rnd(1, 6, seed=2)
    def score(i, j):
        return float(O.rotate_pairs(q, torch.tensor([i]), fr) @ O.rotate_pairs(k, torch.tensor([j]), fr).T)
    assert abs(score(9, 4) - score(105, 100)) < 1e-12 and abs(score(9, 4) - score(9, 5)) > 1e-6
    r = O.rotate_pairs(q, torch.tensor([3]), fr, 1.5)
    assert torch.equal(r[:, 4:], q[:, 4:])                                                       # columns past the rotated ones
    a = 3 * 0.5
    assert abs(float(r[0, 0]) - 1.5 * (float(q[0, 0]) * math.cos(a) - float(q[0, 1]) * math.sin(a))) < 1e-12    # neighbours pair up
    assert abs(float(r[0, 1]) - 1.5 * (float(q[0, 1]) * math.cos(a) + float(q[0, 0]) * math.sin(a))) < 1e-12


def test_oracle_yarn_keeps_fast_pairs_and_slows_the_slow_ones():
    base, dims, factor, original = 10000.0, 16, 4.0, 256.0
    fr, mag = O.yarn_frequencies(base, dims, factor, original, 32.0, 1.0)
    plain, _ = O.plain_frequencies(base, dims)
    turns = original * plain / (2 * math.pi)
    assert abs(mag - (0.1 * math.log(4.0) + 1.0)) < 1e-15
    assert float(turns[0]) > 32 and fr[0] == plain[0]                                           # turns often: untouched
    assert float(turns[-1]) < 1 and abs(float(fr[-1]) - float(plain[-1]) / 4.0) < 1e-18         # hardly turns: divided by the factor
    mid = [i for i in range(8) if plain[i] / 4.0 < fr[i] < plain[i]]
    assert mid and all(fr[i] > fr[i + 1] for i in range(7))


def test_oracle_masks_sinks_and_grouped_heads():
    assert [j for j in range(12) if O.sees_block(9, j, 4)] == [8, 9] and [j for j in range(12) if O.sees_block(8, j, 4)] == [8]
    assert [j for j in range(12) if O.sees_window(9, j, 4)] == [6, 7, 8, 9] and [j for j in range(5) if O.sees_block(3, j, 0)] == [0, 1, 2, 3]
    m, D, Dv = 7, 5, 3
    q, k, v = rnd(m, D, seed=1), rnd(m, D, seed=2), rnd(m, Dv, seed=3)
    plain = O.softmax_attention(q, k, v, list(range(m)), lambda i, j: j <= i, 0.4)
    assert torch.allclose(plain[0], v[0], atol=1e-12)
    sunk = O.softmax_attention(q, k, v, list(range(m)), lambda i, j: j <= i, 0.4, sink=torch.tensor(0.7, dtype=F))
    s0 = float(q[0] @ k[0]) * 0.4
    assert torch.allclose(sunk[0], v[0] * math.exp(s0) / (math.exp(s0) + math.exp(0.7)), atol=1e-12)     # the sink is not scaled, counts once
    far = O.softmax_attention(q, k, v, list(range(m)), lambda i, j: j <= i, 0.4, sink=torch.tensor(-50.0, dtype=F))
    assert torch.allclose(far, plain, atol=1e-12)


def test_oracle_latent_attention_equals_its_folded_form():
    """Keys and values rebuilt from the latent per head (how the oracle writes it) against up-projections folded into the query
    and the output (how the product computes it)."""
    lay = small_shape().layers[2]
    H, D, R, Dv, C = lay.heads, lay.dim, lay.rot_dim, lay.vdim, lay.kv_rank
    Wd = 24
    p = {"m.q": rnd(H * (D + R), Wd, seed=1), "m.dkv": rnd(C + R, Wd, seed=2), "m.dkv.norm": 1 + 0.1 * rnd(C, seed=3), "m.uk": rnd(H * D, C, seed=4),
         "m.uv": rnd(H * Dv, C, seed=5), "m.g": rnd(H * Dv, Wd, seed=6), "m.o": rnd(Wd, H * Dv, seed=7)}
    h = rnd(9, Wd, seed=8)
    y, (c, kr) = O.latent_mixer(h, p, "m.", lay, 1e-5, 0, None)
    fr, mag = O.yarn_frequencies(lay.rot_base, R, lay.rot_factor, lay.yarn_original, lay.yarn_fast, lay.yarn_slow)
    pos = torch.arange(9)
    q = (h @ p["m.q"].T).view(9, H, D + R)
    out = torch.zeros(9, H, Dv, dtype=F)
    for hd in range(H):
        uk, uv = p["m.uk"][hd * D:(hd + 1) * D], p["m.uv"][hd * Dv:(hd + 1) * Dv]
        qq = torch.cat([q[:, hd, :D] @ uk, O.rotate_pairs(q[:, hd, D:], pos, fr, mag)], dim=1)
        o = O.softmax_attention(qq, torch.cat([c, kr], dim=1), c, pos.tolist(), lambda i, j: O.sees_window(i, j, lay.mask), lay.scale)
        out[:, hd] = o @ uv.T
    folded = (out.reshape(9, -1) * torch.sigmoid(h @ p["m.g"].T)) @ p["m.o"].T
    assert torch.allclose(folded, y, atol=1e-10)


def test_oracle_matrix_memory_in_closed_form():
    """With the running maximum taken out, token t's numerator is sum_j exp(F_t - F_j + i_j) (q_t . k_j) v_j, F the running sum of
    the log forget gates; the maximum only rescales numerator and denominator alike, except through the floor exp(-m)."""
    n, H, D, Dv = 8, 1, 3, 2
    q, k, v = rnd(n, H, D, seed=1), rnd(n, H, D, seed=2), rnd(n, H, Dv, seed=3)
    li, lf = rnd(n, H, seed=4), -rnd(n, H, seed=5).abs()
    out, (S, nv, m) = O.matrix_memory(q, k, v, li, lf)
    Fs = torch.cumsum(lf[:, 0], 0)
    for t in (0, 3, 7):
        wts = torch.stack([torch.exp(Fs[t] - Fs[j] + li[j, 0]) * (q[t, 0] @ k[j, 0]) for j in range(t + 1)])
        num = (wts.unsqueeze(1) * v[:t + 1, 0]).sum(0)
        mt = 0.0                                              # the running maximum, starting from 0
        for j in range(t + 1):
            mt = max(float(lf[j, 0]) + mt, float(li[j, 0]))
        den = max(abs(float(wts.sum())), 1.0) * math.exp(-mt) + 1e-6    # (both sides of the max carry exp(-m): |n.q| e^-m vs e^-m)
        assert torch.allclose(out[t, 0], num * math.exp(-mt) / den, atol=1e-10), t
    a, st = O.matrix_memory(q[:5], k[:5], v[:5], li[:5], lf[:5])
    b, st2 = O.matrix_memory(q[5:], k[5:], v[5:], li[5:], lf[5:], st)
    assert torch.allclose(torch.cat([a, b]), out, atol=1e-12) and torch.allclose(st2[0], S, atol=1e-12) and torch.allclose(st2[2], m, atol=1e-12)
    assert O.soft_cap(torch.tensor(100.0, dtype=F), 9.0) < 9.0 and O.soft_cap(torch.tensor(3.0, dtype=F), 0.0) == 3.0


def test_oracle_gated_sublayer_and_feed_forward():
    Wd, ff = 6, 5
    p = {"l.norm2": 1 + 0.1 * rnd(Wd, seed=1), "l.norm2b": 1 + 0.1 * rnd(Wd, seed=2), "l.rg2": rnd(Wd, Wd, seed=3), "l.rg2.b": rnd(Wd, seed=4),
         "m.gate": rnd(ff, Wd, seed=5), "m.gate.b": rnd(ff, seed=6), "m.up": rnd(ff, Wd, seed=7), "m.up.b": rnd(ff, seed=8),
         "m.down": rnd(Wd, ff, seed=9), "m.down.b": rnd(Wd, seed=10)}
    x = rnd(4, Wd, seed=11)
    h = O.unit_rms(x, 1e-5) * p["l.norm2"]
    y = (torch.relu(h @ p["m.gate"].T + p["m.gate.b"]) * (h @ p["m.up"].T + p["m.up.b"])) @ p["m.down"].T + p["m.down.b"]
    assert torch.allclose(O.dense_ff(h, p, "m."), y, atol=1e-12)
    t = y * torch.sigmoid(h @ p["l.rg2"].T + p["l.rg2.b"])
    want = x + t / torch.sqrt(t.pow(2).mean(-1, keepdim=True) + 1e-5) * p["l.norm2b"]
    assert torch.allclose(O.gated_sublayer(x, lambda hh: O.dense_ff(hh, p, "m."), p, "l.", "2", 1e-5), want, atol=1e-12)
    z = torch.tensor([-1.0, 0.5, 2.0], dtype=F)
    assert torch.allclose(O.activation("gelu_tanh")(z), 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3))))


@pytest.mark.parametrize("requests,heads,dim,vdim,tokens,segments", [
    # where one of the two ways through the matrix memory was measured to be the faster by 8 % or more
    (1, 16, 128, 128, 8, False), (1, 16, 128, 128, 16, True), (8, 8, 128, 128, 8, False), (8, 16, 128, 128, 8, False), (8, 16, 128, 128, 24, True),
    (32, 8, 128, 128, 16, False), (8, 32, 128, 128, 16, False), (8, 32, 128, 128, 32, True), (40, 16, 128, 128, 15, True), (80, 16, 128, 128, 11, False),
    (24, 12, 128, 64, 22, False), (24, 12, 128, 64, 40, True), (1, 16, 64, 64, 10, False), (1, 16, 64, 64, 20, True), (32, 16, 64, 64, 24, False),
    (40, 8, 64, 64, 28, False), (32, 32, 64, 64, 32, False), (32, 4, 64, 64, 32, True)])
def test_few_tokens_go_through_the_matrix_memory_one_by_one(requests, heads, dim, vdim, tokens, segments):
    from promptcache_amd.model.fivesun_hip import FivesunHIP
    assert (tokens > FivesunHIP._few_tokens(requests, heads, dim, vdim)) == segments


@pytest.mark.parametrize("heads,dim,vdim,width,dtype,fits", [
    (16, 128, 128, 2048, torch.bfloat16, True), (16, 128, 128, 2048, torch.float32, True), (2, 16, 24, 64, torch.float32, True), (2, 16, 24, 64, torch.bfloat16, False),
    (3, 128, 128, 2048, torch.bfloat16, False), (4, 136, 64, 512, torch.bfloat16, False), (4, 64, 60, 512, torch.float32, False), (4, 64, 64, 508, torch.bfloat16, False)])
def test_layers_and_calls_share_the_rule_of_what_goes_in_segments(heads, dim, vdim, width, dtype, fits):
    """What a model decides from a layer's sizes is what the call says of the same columns."""
    from types import SimpleNamespace
    from promptcache_amd import _blocks as B
    from promptcache_amd.model.fivesun_hip import FivesunHIP
    layer = FivesunLayer("mlstm", heads=heads, kv_heads=heads, dim=dim, vdim=vdim, ff=16)
    assert FivesunHIP._mlstm_fits(SimpleNamespace(dtype=dtype, W=width), layer) == fits
    at = [0, heads * dim, 2 * heads * dim]
    gate = 2 * heads * dim + heads * vdim + 2 * heads
    n = gate + heads * vdim + width
    es = torch.empty(0, dtype=dtype).element_size()
    mem = torch.empty(2 * n + 16, dtype=dtype)
    mem = mem[(-mem.data_ptr() % 16) // es:]
    assert B.mlstm_prompt_fits(dim, vdim, n, [mem[a:] for a in at], mem[gate:], 64) == fits


# ---- launches of a step whose norm rides in a projection -------------------------------------------------------------------------
class _NoLaunch:
    """The blocks library with every call that would launch answered with "done"; what pcb_norm_linear is given is kept."""

    def __init__(self, lib, launches, seen):
        self.lib, self.launches, self.seen, self.names = lib, launches, seen, []

    def __getattr__(self, name):
        if name not in self.launches:
            return getattr(self.lib, name)

        def call(*args):
            self.names.append(name)
            if name == "pcb_norm_linear":
                self.seen.append([None if a is None else type(a._obj).from_buffer_copy(a._obj) for a in args[:3]])
            return 0
        return call


def no_launches(monkeypatch):
    """Steps on the host whose launches do nothing; -> what pcb_norm_linear is given, call by call."""
    from promptcache_amd import _blocks as B
    launches = {n for n, (_, args) in B.SIGNATURES.items() if args and args[-1] is ctypes.c_void_p}
    seen = []
    monkeypatch.setattr(B, "_lib", _NoLaunch(B.load(), launches, seen))
    monkeypatch.setattr(B, "_stream", lambda: 0)
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)               # (there is no device here: the tensors lie on the host)
    return seen


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 3])
def test_a_norms_rows_lie_apart_from_what_its_launch_stores(monkeypatch, rows, dtype):
    """A layer without a feed-forward leaves its residual gate in its projected rows: the next layer's products, in whose launch the gate is read, store elsewhere."""
    from promptcache_amd.model.fivesun_hip import FivesunHIP
    att = dict(heads=4, kv_heads=2, dim=16, vdim=16, scale=0.25, mask=0, rot_base=100.0, rot_dims=16, rot_factor=1.0, v_mix=True)
    lat = dict(heads=2, kv_heads=1, dim=16, vdim=16, kv_rank=32, rot_dim=16, rot_dims=16, scale=0.2, mask=9, rot_base=50.0, rot_factor=1.0)
    mem = dict(heads=2, kv_heads=2, dim=16, vdim=16, gate_cap=4.0)
    s = FivesunShape(vocab_size=60, hidden_size=512, norm_eps=1e-5, embed_scale=3.5, layers=[
        FivesunLayer("attention", **att), FivesunLayer("attention", **att), FivesunLayer("latent_attention", **lat), FivesunLayer("mlstm", **mem),
        FivesunLayer("attention", ff=64, **att), FivesunLayer("mlstm", **mem), FivesunLayer("mlstm", **mem), FivesunLayer("latent_attention", **lat)])
    seen = no_launches(monkeypatch)
    m = FivesunHIP(s, W.make_fivesun_weights(s, seed=1), device="cpu", dtype=dtype)
    m.use_graphs = False
    ar = m.new_arena(rows, 8)
    m.forward_rows(ar, [ar.alloc() for _ in range(rows)], [[5]] * rows)
    assert len(seen) == len(s.layers) + 1
    es = 2 if dtype == torch.bfloat16 else 4
    for n, a, b in seen:
        span = lambda p, ld, cols, size: (p, p + ((rows - 1) * ld + cols) * size)       # noqa: E731
        read = [span(p, ld, 512, size) for p, ld, size in ((n.x, 512, 4), (n.y, 512, 4), (n.gate, n.ldg, es)) if p]
        stored = [span(n.x_out, 512, 512, 4)] + [span(q.y, q.ldy, q.N, es) for q in (a, b) if q is not None]
        for lo, hi in read:
            assert all(hi <= at or end <= lo for at, end in stored)


def test_rows_of_a_few_row_step_only_have_their_second_scratch(monkeypatch):
    """What exists so that a norm may ride in a projection's launch is not allocated for steps in which it cannot."""
    from promptcache_amd.model.fivesun_hip import FivesunHIP
    no_launches(monkeypatch)
    att = dict(heads=4, kv_heads=2, dim=16, vdim=16, scale=0.25, mask=0, rot_base=100.0, rot_dims=16, rot_factor=1.0)
    s = FivesunShape(vocab_size=60, hidden_size=512, norm_eps=1e-5, embed_scale=3.5, layers=[FivesunLayer("attention", **att), FivesunLayer("attention", **att)])
    m = FivesunHIP(s, W.make_fivesun_weights(s, seed=1), device="cpu")
    m.use_graphs = False
    ar = m.new_arena(1, 300)
    slot = ar.alloc()
    m.forward_rows(ar, [slot], [[5] * 200])
    assert not {"x_next", "mix_in_next"} & set(m._buf)
    m.forward_rows(ar, [slot], [[5]])
    assert m._buf["x_next"].numel() == 1024 and m._buf["mix_in_next"].numel() < m._buf["mix_in"].numel()


@pytest.mark.parametrize("dtype,rows,reach,step", [
    (torch.bfloat16, 1, 60000, True), (torch.bfloat16, 8, 60000, True), (torch.bfloat16, 64, 8000, True), (torch.bfloat16, 64, 8100, False), (torch.bfloat16, 128, 4000, False),
    (torch.bfloat16, 192, 2000, True), (torch.bfloat16, 512, 2000, False), (torch.bfloat16, 1024, 1000, True), (torch.float32, 128, 4000, False),
    (torch.float32, 128, 8000, False), (torch.float32, 512, 1000, True), (torch.float32, 64, 2000, True)])
def test_steps_over_latents_take_one_launch_where_that_is_the_faster(monkeypatch, dtype, rows, reach, step):
    """The rule by rows and reach, and the launches of a step on either side of it."""
    from promptcache_amd import _blocks as B
    from promptcache_amd.model.fivesun_hip import FivesunHIP
    lat = dict(heads=2, kv_heads=1, dim=16, vdim=16, kv_rank=32, rot_dim=16, rot_dims=16, scale=0.2, mask=0, rot_base=50.0, rot_factor=1.0)
    s = FivesunShape(vocab_size=60, hidden_size=64, norm_eps=1e-5, layers=[FivesunLayer("latent_attention", **lat)])
    no_launches(monkeypatch)
    m = FivesunHIP(s, W.make_fivesun_weights(s, seed=1), device="cpu", dtype=dtype)
    m.use_graphs = False
    splits = m._step_splits(rows, 1, 16, reach, 768, rows <= 64)
    assert m._latent_step(rows, 1, reach, splits) == step
    m._latent_step = lambda *a: step
    ar = m.new_arena(2, 8)
    m.forward_rows(ar, [ar.alloc(), ar.alloc()], [[5], [6]])
    assert ("pcb_attn_step" in B._lib.names) == step and ("pcb_attn_latent" in B._lib.names) != step


def test_results_over_the_rows_of_a_norm_go_apart(monkeypatch):
    """pcb_norm_linear does not take products that store over what the norm reads, and refuses such an x_out; decided on the host, nothing is launched."""
    from promptcache_amd import _blocks as B
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    M, K, N = 2, 512, 640
    x, y, gate, gain = torch.zeros(M, K), torch.zeros(M, K), torch.zeros(M, K + 128, dtype=torch.bfloat16), torch.ones(K)
    out, h, w = torch.zeros(M, K), torch.zeros(M, K, dtype=torch.bfloat16), torch.zeros(N, K, dtype=torch.bfloat16)
    P, Q = torch.zeros(M, N, dtype=torch.bfloat16), torch.zeros(M, N, dtype=torch.bfloat16)
    room = torch.zeros(4 * M * K)                                    # streams, and what lies around them

    def asked(a, b=None, x_out=out, streams=None):
        n = B.RowNormArgs(ctypes.sizeof(B.RowNormArgs), x.data_ptr(), 0, None, 0, None, None, 0, 1.0, y.data_ptr(), gate.data_ptr() + 256, K + 128, gain.data_ptr(),
                          gain.data_ptr(), gain.data_ptr(), x_out.data_ptr(), 1e-5)
        if streams is not None:
            n.x, n.x_stride, n.coef, n.n_terms, n.y, n.gate, n.ldg, n.post_gain = streams.data_ptr(), M * K, gain.data_ptr(), 2, None, None, 0, None
        return B.load().pcb_norm_linear_takes(ctypes.byref(n), ctypes.byref(a), None if b is None else ctypes.byref(b))

    def product(to):
        return B.linear_args(h, w, to, M=M)
    bf = lambda t: t.view(torch.bfloat16).view(-1)                   # noqa: E731
    assert asked(product(P)) == 0 and asked(product(P), product(Q)) == 0
    assert asked(product(bf(x)[:M * N].view(M, N))) == B.NOT_TAKEN and asked(product(bf(y)[:M * N].view(M, N))) == B.NOT_TAKEN
    assert asked(product(gate.view(-1)[:M * N].view(M, N))) == B.NOT_TAKEN
    assert asked(product(P), product(gate.view(-1)[:M * N].view(M, N))) == B.NOT_TAKEN
    assert asked(product(bf(out)[:M * N].view(M, N))) == B.NOT_TAKEN
    tail = bf(room)
    # two streams of M x K: their last element counts, what begins behind it does not; an fp32 result by its own size
    assert asked(product(tail[4 * M * K:4 * M * K + M * N].view(M, N)), streams=room) == 0
    assert asked(product(tail[4 * M * K - 8:4 * M * K - 8 + M * N].view(M, N)), streams=room) == B.NOT_TAKEN
    assert asked(product(tail[:M * N].view(M, N)), streams=room[M * N // 2:]) == 0
    assert asked(product(room[:M * N].view(M, N)), streams=room[M * N // 2:]) == B.NOT_TAKEN
    for over in (x, y, gate.view(torch.float32)):
        assert asked(product(P), x_out=over) == -2001
    assert asked(product(P), x_out=room[M * K:], streams=room) == -2001 and asked(product(P), x_out=room[2 * M * K:], streams=room) == 0


@pytest.mark.parametrize("splits,up,off", [(1, True, 4), (0, True, 8), (2, False, 4), (65, False, 0), (65, True, 0), (1, True, None), (3, False, None)])
def test_scratch_of_a_decoding_step_is_checked_wherever_it_is_used(splits, up, off):
    """Whole 16 bytes, up to 64 runs; refused on the host (no device is needed)."""
    from promptcache_amd import _blocks as B
    room = torch.zeros(4096)
    at = room.data_ptr() // 16 * 16 + 16
    a = B.AttnStepArgs(ctypes.sizeof(B.AttnStepArgs), B.F32)
    a.p = a.q = a.tiles = a.k = a.v = a.out = a.freqs = at
    a.ldp, a.ldq, a.ldo, a.n_rows, a.H, a.Hkv, a.dim, a.vdim, a.latent, a.rot_dims = 256, 64, 64, 1, 1, 1, 48, 32, 1, 16
    a.k_row_stride = a.v_row_stride = 48
    a.n_splits, a.part = splits, None if off is None else at + off
    if up:
        a.up, a.up_dim, a.up_gate, a.ld_up_gate = at, 64, at, 64
    assert B.load().pcb_attn_step_fits(B.F32, 1, 1, 48, 32, 16, 1)
    assert B.load().pcb_attn_step(ctypes.byref(a), None) == -2001 and b"scratch" in B.load().pcb_last_error_string()
