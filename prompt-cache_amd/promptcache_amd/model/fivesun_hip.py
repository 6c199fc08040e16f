"""Fivesun forward pass on MI355X (``config.FivesunShape`` says what the design is).

Like ``dibizen_hip.DibizenHIP`` this model keeps plain row-major tensors in one element type E -- bfloat16 (serving: matrix
products on the bf16 matrix cores, fp32 accumulation) or float32 (everything in true 32-bit) -- runs on the building blocks of
``libpromptcache_blocks.so`` (``_blocks.py``) and steps over FLAT rows: the new tokens of all requests of a step one after
another, each request continuing from what its slot of the ``SlotArena`` holds.  Nothing is padded, and a row reads nothing but
its own slot, so a request's numbers do not depend on the rest of the step.

What a slot holds differs by layer: an attention layer keeps rows ``key | value`` (keys normed and rotated, values normed and
blended), a latent-attention layer ONE row per token -- the normed latent followed by the rotated shared key part --, an mLSTM
layer its fp32 matrix memory, normaliser and running maximum.

The residual x is fp32.  Sublayer by sublayer (f = mixer or feed-forward, each between a norm before and a norm after it):

    h = rms(x) g_before                          t = f(h) * sigmoid(W_r h + b_r)          x <- x + rms(t) g_after

``pcb_post_norm`` applies a finished sublayer's t and takes the next sublayer's norm in one launch; the sigmoid gate rides in the
same projection as the mixer's inputs (or is one projection beside the feed-forward's).

    attention   q | k | v | g | r = ONE projection (sigmoid on g | r); pcb_head_prep: per-head RMS norms, rotary pairs (angles as
                float64 products), value blend with the first blending layer's values, ``key | value`` rows into the slot's cache;
                keys of the query's own block of positions only, exp(sink_h) in the denominator, one gate per head: tiles of
                queries where requests bring many tokens for their context (pcb_attn_prompt), single rows elsewhere (pcb_attn_rows)
    latent      q | down | g | r = ONE projection; pcb_head_prep: the latent normed, the shared key part and the queries' rotated
                parts turned (YaRN frequencies), latent | key part into the slot's row.  A request that brings many tokens may have the
                keys and values of all heads rebuilt from the latents (pcb_linear) and attends in tiles (pcb_attn_prompt, the shared
                key part read from the cached rows, times sigmoid(g)); for the others the up-projections are folded into the query
                and the output: q'_h = W_uk,h^T q_h, attention of [q'_h | q_rot,h] over the cached rows with the latent itself as
                value (pcb_attn_latent, sliding window), o_h = W_uv,h (.), times sigmoid(g).  Heads too wide for the tiles fold always
    mlstm       q | k | v | i | f | g | r = ONE projection; the gated matrix memory, per-head unit RMS, gain, sigmoid(g): in segments on the
                matrix cores (pcb_mlstm_prompt), one token per request (pcb_mlstm_step), or, for sizes these do not take, token by
                token (pcb_mlstm, pcb_gated_norm)
    dense ff    act(W_gate h + b) * (W_up h + b) in one projection's epilogue, then W_down (.) + b

and the logits are ``head . rms(x) g`` for the rows that were asked for.
"""
from __future__ import annotations

import math
import os
from collections import Counter
from typing import Dict, Optional, Sequence

import numpy as np
import torch

from .. import _blocks as B
from .config import FivesunShape
from .kv_arena import SlotArena
from .slot_model import SlotKV, SlotModel, StepRows  # noqa: F401

ACTS = {"relu": B.ACT_RELU, "silu": B.ACT_SILU, "gelu_tanh": B.ACT_GELU_TANH}


def rotary_frequencies(base: float, dims: int, factor: float = 1.0, original: float = 0.0, fast: float = 32.0, slow: float = 1.0):
    """float64 frequencies of the ``dims / 2`` rotated column pairs and the factor on cos and sin.  Plain: base^(-2i/dims) / factor.
    With ``original`` > 0 (YaRN): pairs that complete more than ``fast`` turns over ``original`` positions keep their frequency,
    those with fewer than ``slow`` turns are divided by ``factor``, a linear ramp over the pair index between them; the rotated
    vector grows by 0.1 ln(factor) + 1."""
    f = np.asarray([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=np.float64)
    if original <= 0:
        return f / factor, 1.0

    def pair_of(turns):
        return dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo, hi = max(math.floor(pair_of(fast)), 0), min(math.ceil(pair_of(slow)), dims - 1)
    ramp = np.clip((np.arange(dims // 2, dtype=np.float64) - lo) / max(hi - lo, 0.001), 0.0, 1.0)
    return f / factor * ramp + f * (1.0 - ramp), 0.1 * math.log(factor) + 1.0


class FivesunHIP(SlotModel):
    GRAPH_MAX_ROWS = 64
    # Tokens of a segment of the mLSTM layers.  Where all of them fit the matrix cores' kernels (_mlstm_fits), a step that brings a request more than
    # _few_tokens() runs them in segments, else one that brings more than SEGMENT; the others go token by token.
    SEGMENT = int(os.environ.get("PC_FS_SEGMENT", "64"))
    MAX_SEGMENTS = 128      # (segments grow beyond SEGMENT tokens rather than exceed this many per request)
    PROMPT_ROWS = int(os.environ.get("PC_FS_PROMPT_ROWS", "16"))   # a request that brings fewer tokens than this attends row by row (see _tiled)
    # Rebuilt keys and values that lie in memory at a time: beyond it heads take turns, which leaves part of the chip idle (eight requests of 256
    # tokens behind 8 000, 541 MB: 3 350 us in one turn, 4 023 in three).  1 GB is 131 k rows of 16 heads of 128 + 128 columns.
    REBUILD_BYTES = 1 << 30

    def __init__(self, shape: FivesunShape, weights: Dict[str, torch.Tensor], device="cuda:0", dtype=torch.bfloat16,
                 decode_headroom: int = 256):
        if dtype not in (torch.bfloat16, torch.float32):
            raise ValueError("Fivesun runs in bfloat16 or float32")
        B.load()                                   # fail loudly (or build once) before anything else
        shape.check()
        self.config = shape
        self.device = torch.device(device)
        self.dtype = dtype
        self.decode_headroom = decode_headroom
        self.L = len(shape.layers)
        self.W, self.V = shape.hidden_size, shape.vocab_size
        if self.W > 16384:
            raise ValueError(f"width up to 16384 (got {self.W})")
        dev, W = self.device, self.W

        def e(name):                               # element-type tensor (projections and their biases)
            return weights[name].to(device=dev, dtype=dtype).contiguous()

        def f(name):                               # fp32 tensor (norm gains, sinks, blend weights)
            return weights[name].to(device=dev, dtype=torch.float32).contiguous()

        def zeros(n):
            return torch.zeros(n, dtype=dtype, device=dev)

        self.embed, self.final_norm, self.head = e("embed"), f("final.norm"), e("head")
        self.first_v_mix = shape.first_v_mix
        self.layers = []
        for i, l in enumerate(shape.layers):
            p, m = f"l{i}.", f"l{i}.mix."
            ent = dict(cfg=l, norm1=f(p + "norm1"), norm1b=f(p + "norm1b"))
            rg, rgb = e(p + "rg1"), e(p + "rg1.b")
            if l.kind == "attention":
                if l.dim > 384 or l.vdim > 256:
                    raise ValueError(f"layer {i}: attention heads take up to 384 key and 256 value columns (got {l.dim} / {l.vdim})")
                HD, GD, GV = l.heads * l.dim, l.kv_heads * l.dim, l.kv_heads * l.vdim
                fr, mag = rotary_frequencies(l.rot_base, l.rot_dims, l.rot_factor) if l.rot_dims else (np.zeros(0), 1.0)
                ent.update(w_in=torch.cat([e(m + "q"), e(m + "k"), e(m + "v"), e(m + "g"), rg], dim=0).contiguous(),
                           b_in=torch.cat([zeros(HD + GD + GV + l.heads), rgb]).contiguous(), act_from=HD + GD + GV,
                           q_gain=f(m + "q.norm"), k_gain=f(m + "k.norm"), sink=f(m + "sink"), wo=e(m + "o"),
                           blend=f(m + "vmix").reshape(1) if (l.v_mix and i != self.first_v_mix) else None,
                           freqs=torch.from_numpy(fr).to(dev) if l.rot_dims else None, rot_mag=mag)
            elif l.kind == "latent_attention":
                C, R = l.kv_rank, l.rot_dim
                if C + R > 384 or C > 256:
                    raise ValueError(f"layer {i}: a latent of up to 256 columns plus a rotated part within 384 together (got {C} + {R})")
                HQ, HV = l.heads * (l.dim + R), l.heads * l.vdim
                fr, mag = rotary_frequencies(l.rot_base, R, l.rot_factor, l.yarn_original, l.yarn_fast, l.yarn_slow) if R else (np.zeros(0), 1.0)
                # (the tiled attention takes heads of up to 256 key and 256 value columns)
                ent.update(w_in=torch.cat([e(m + "q"), e(m + "dkv"), e(m + "g"), rg], dim=0).contiguous(),
                           b_in=torch.cat([zeros(HQ + C + R + HV), rgb]).contiguous(), act_from=HQ + C + R,
                           prompts=l.dim + R <= 256 and l.vdim <= 256, w_kv=torch.cat([e(m + "uk"), e(m + "uv")], dim=0).contiguous(),
                           c_gain=f(m + "dkv.norm"), wo=e(m + "o"),
                           # per head: the key up-projection transposed ([C, dim]: it maps a query to the latent's columns) and the
                           # value up-projection as stored ([vdim, C])
                           w_abs=e(m + "uk").view(l.heads, l.dim, C).transpose(1, 2).contiguous(),
                           w_uv=e(m + "uv").view(l.heads, l.vdim, C).contiguous(),
                           freqs=torch.from_numpy(fr).to(dev) if R else None, rot_mag=mag)
            else:
                if l.dim > 256:
                    raise ValueError(f"layer {i}: mLSTM heads take up to 256 key columns (got {l.dim})")
                HD, HV, H = l.heads * l.dim, l.heads * l.vdim, l.heads
                ent.update(w_in=torch.cat([e(m + "q"), e(m + "k"), e(m + "v"), e(m + "i"), e(m + "f"), e(m + "g"), rg], dim=0).contiguous(),
                           b_in=torch.cat([zeros(2 * HD + HV), e(m + "i.b"), e(m + "f.b"), zeros(HV), rgb]).contiguous(),
                           act_from=2 * HD + HV + 2 * H, gain=f(m + "norm"), wo=e(m + "o"))
            if l.ff:
                if l.act not in ACTS:
                    raise ValueError(f"layer {i}: unknown activation {l.act!r}")
                q = p + "mlp."
                ent.update(norm2=f(p + "norm2"), norm2b=f(p + "norm2b"), rg2=e(p + "rg2"), rg2b=e(p + "rg2.b"),
                           w_gate=e(q + "gate"), b_gate=e(q + "gate.b"), w_up=e(q + "up"), b_up=e(q + "up.b"),
                           w_down=e(q + "down"), b_down=e(q + "down.b"))
            self.layers.append(ent)
        self._buf = {}
        self.default_arena: Optional[SlotArena] = None
        self.use_graphs = os.environ.get("PC_FS_GRAPHS", "1") != "0"      # one-token steps replay a captured hipGraph
        self._graphs = {}
        self.max_graphs = 16
        # cache offsets of a row, one table per distinct (heads, columns) of the planes
        self._sigs = sorted({(l.kv_heads, l.dim + l.vdim) for l in shape.layers if l.kind == "attention"} |
                            {(1, l.kv_rank + l.rot_dim) for l in shape.layers if l.kind == "latent_attention"})
        latent = [ent for ent in self.layers if ent["cfg"].kind == "latent_attention"]
        self._folds = any(not ent["prompts"] for ent in latent)
        # what _tiled weighs: (heads, workgroups a row takes in the kernels of single rows, reach, columns rebuilt per key and head), how many layers
        self._att = Counter((l.heads, l.kv_heads * -(-l.heads // (16 * l.kv_heads)), l.mask, 0) for l in shape.layers if l.kind == "attention" and l.dim <= 256)
        self._lat = Counter((l.heads, -(-l.heads // 16), l.mask, l.kv_rank * (l.dim + l.vdim)) for l in (ent["cfg"] for ent in latent if ent["prompts"]))
        # positions behind a request's first new token whose keys its rebuilding layers need (0: all of them)
        reach = [mask for _, _, mask, _ in self._lat]
        self._reach = 0 if not reach or min(reach) <= 0 else max(reach)
        self._wide = any(ent["cfg"].kind == "attention" and ent["cfg"].dim > 256 for ent in self.layers)
        self._chunks = all(self._mlstm_fits(l) for l in shape.layers if l.kind == "mlstm")
        self._max_heads = max(l.heads for l in shape.layers)

    @staticmethod
    def _few_tokens(requests, heads, dim, vdim):
        """Up to how many tokens a request (the longest of the step) the memory is faster token by token.  That costs a fixed time a token until its
        workgroups (one per request and head) are more than fit the chip at once; segments cost the same for 2 as for 16 tokens, and in proportion to
        requests x heads.  us, token by token / in segments, heads of 128: 16 of them 8 tokens 22.1 / 24.6, 10 25.1 / 24.8; 128 13 tokens 29.2 / 31.3, 16
        31.5 / 31.3; 256 20 tokens 38.7 / 44.6, 24 42.7 / 44.6; 640 13 85 / 67 (bf16), 1280 13 139 / 167 (fp32); heads of 64: 16 of them 14 tokens
        20.4 / 21.1, 16 21.7 / 21.1; 320 28 tokens 34 / 36 (fp32), 1024 32 tokens 54 / 76; 128 x 64, 288 of them 22 tokens 41 / 47."""
        n = requests * heads
        if dim <= 64:
            return 15 + n // 24
        if vdim > 64 and n > 256:
            return 12 if n <= 1024 else 14
        return min(22, 8 + n * dim * dim // (1 << 18))

    def _mlstm_fits(self, l):
        """Whether an mLSTM layer's columns of the step's projection (q | k | v | i | f | gate | residual gate) are what ``B.mlstm_prompt`` takes."""
        HD, HV, es = l.heads * l.dim, l.heads * l.vdim, 2 if self.dtype == torch.bfloat16 else 4
        gate = 2 * HD + HV + 2 * l.heads
        return B.mlstm_prompt_takes(l.dim, l.vdim, gate + HV + self.W, es, (0, es * HD, 2 * es * HD), es * gate, 1)

    # ---- cache and state -------------------------------------------------------------------------------------------------------
    def new_arena(self, slots: int, cap: int) -> SlotArena:
        dims, states = [], []
        for l in self.config.layers:
            if l.kind == "attention":
                dims.append((l.kv_heads, l.dim + l.vdim)); states.append([])
            elif l.kind == "latent_attention":
                dims.append((1, l.kv_rank + l.rot_dim)); states.append([])
            else:
                dims.append((0, 0))
                states.append([((B.mlstm_state_floats(l.heads, l.dim, l.vdim),), torch.float32)])
        return SlotArena(dims, slots, cap, self.device, self.dtype, states=states)

    def kv_bytes_per_token(self) -> int:
        es = 2 if self.dtype == torch.bfloat16 else 4
        return sum(l.kv_heads * (l.dim + l.vdim) if l.kind == "attention" else (l.kv_rank + l.rot_dim if l.kind == "latent_attention" else 0)
                   for l in self.config.layers) * es

    def _tiled(self, layers, cand, counts, starts):
        """Which of the requests ``cand`` attend in tiles of queries in ``layers``; the others go row by row.

        A tile walks its request's keys by itself, so tiles are as slow as the longest context among them, however little of the chip they
        fill; rows are cut into runs of keys and cost the same each.  In units of a tile's block of 64 keys (2.25 us; fp32 6.6): a row costs
        1 / 700 a block and workgroup, 470 tiles run at a time (fp32 320), a latent layer's tile block 1.16, its rebuilt block
        heads * rank * (key + value columns) / 6.5e6, its folded row heads / 4400 for the products around it.  Tiled are the requests up to the
        context length that makes the sum cheapest.  us, heads of 128, rows / tiles, keys x tokens: 16 heads over 4, 1 024 x 64 23 / 41, x 256
        79 / 47, 8 000 x 64 121 / 296, x 256 401 / 290, 30 000 x 16 119 / 1 030, x 256 1 384 / 1 039, eight requests of 8 000 x 16 235 / 287, x 64
        769 / 290; latent of 192, folded / rebuilt: 8 000 x 64 49 / 375, x 512 281 / 381, eight requests of 8 000 x 64 282 / 684, x 256 836 / 723."""
        if not cand or not layers:
            return []
        order = sorted(cand, key=lambda b: starts[b] + counts[b])
        shortest, longest = starts[order[0]] + counts[order[0]], starts[order[-1]] + counts[order[-1]]
        if longest <= 512:
            return cand                            # (a dozen us either way, which the host's part of the step covers)
        if all(not l[3] and sum(counts[b] for b in cand) * l[1] * shortest >= 1400 * longest for l in layers):
            return cand                            # (rows would cost twice the longest context's tile)
        at_a_time = 470.0 if self.dtype == torch.bfloat16 else 320.0
        cost = [0.0] * (len(order) + 1)            # of the first k in tiles
        for (heads, groups, mask, rebuilt), n in layers.items():
            unit = 1.16 if rebuilt else 1.0
            rows = [counts[b] * (groups * min(starts[b] + 0.5 * counts[b], mask or math.inf) / (64 * 700) + (heads / 4400 if rebuilt else 0.0)) for b in order]
            rest, longest, all_tiles, rebuild = sum(rows), 0.0, 0.0, 0.0
            cost[0] += n * (rest + 3.0)            # (3 and 2: the launches)
            for k, b in enumerate(order):
                keys = min(starts[b] + counts[b], mask + 64 if mask else math.inf)
                blocks = -(-keys // 64) * unit
                longest = max(longest, blocks)
                all_tiles += -(-counts[b] // 64) * blocks * heads / at_a_time
                rebuild += min(starts[b] + counts[b], mask + counts[b] if mask else math.inf) / 64 * heads * rebuilt / 6.5e6
                rest -= rows[k]
                cost[k + 1] += n * (max(longest, all_tiles) + rebuild + 2.0 + (rest + 3.0 if k + 1 < len(order) else 0.0))
        best = min(range(len(cost)), key=lambda k: (cost[k], -k))
        return sorted(order[:best])

    # ---- one step ------------------------------------------------------------------------------------------------------------
    @torch.inference_mode()
    def forward_rows(self, arena: SlotArena, slots: Sequence[int], tokens: Sequence[Sequence[int]],
                     want: Optional[Sequence[Sequence[int]]] = None, num_layers: Optional[int] = None,
                     return_streams: bool = False):
        """Append ``tokens[b]`` behind slot ``slots[b]`` for every b, and return fp32 logits ``[n_wanted, vocab]`` for the places
        ``want[b]`` (indices into ``tokens[b]``; default: each request's last token), in request order.
        ``return_streams``: also the residual stream after each layer, fp32 ``[layers, rows, width]`` (for tests)."""
        dev = self.device
        if not tokens and not slots:
            return torch.empty((0, self.V), dtype=torch.float32, device=dev)
        st = StepRows(arena, slots, tokens, want, self.V)
        T, R, cap, row0, counts, starts = st.T, st.R, arena.cap, st.row0, st.counts, st.starts
        graphed = (self.use_graphs and T <= self.GRAPH_MAX_ROWS and all(c == 1 for c in counts) and num_layers is None
                   and not return_streams)
        picked, want_rows = None, st.want_rows
        if graphed:
            if any(len(ws) != 1 for ws in st.want):
                picked = [b for b, ws in enumerate(st.want) for _ in ws]
            want_rows = np.arange(T, dtype=np.int32)
        reqs = np.asarray([(s, s0, c, int(row0[b])) for b, (s, s0, c) in enumerate(zip(slots, starts, counts))], dtype=np.int32)

        # attention: tiles of neighbouring queries for requests that bring many tokens, single rows for the others.  (A captured step has single
        # rows only: its launches are those of any step of as many requests.)
        cand = [] if graphed else [b for b, c in enumerate(counts) if c >= self.PROMPT_ROWS]
        big, rebuilt = self._tiled(self._att, cand, counts, starts), self._tiled(self._lat, cand, counts, starts)
        # the oldest key that the rebuilding layers need (a whole number of the kernel's blocks of keys)
        oldest = [max(0, s0 - self._reach + 1) // 64 * 64 if self._reach else 0 for s0 in starts] if rebuilt else []
        tile = 64
        if self.dtype == torch.bfloat16 and sum(-(-counts[b] // 128) for b in big or rebuilt) * self._max_heads >= 512:
            tile = 128
        none = np.zeros(0, np.int32)
        rows = np.empty((T, 4), dtype=np.int32)                 # every row by itself
        rows[:, 0], rows[:, 1], rows[:, 2], rows[:, 3] = st.row_slot, st.row_pos, 1, np.arange(T, dtype=np.int32)

        def others(which):                                      # the flat rows of the other requests
            if not which:
                return slice(None)
            mine = np.zeros(R, dtype=bool)
            mine[which] = True
            return np.flatnonzero(~np.repeat(mine, counts))

        def tiles_of(which, base):
            t = [(base[b], starts[b] + q, min(tile, counts[b] - q), int(row0[b]) + q) for b in which for q in range(0, counts[b], tile)]
            t.sort(key=lambda t: t[1] + t[2])     # (longer contexts behind the shorter ones: the kernel starts from the last tile)
            return np.asarray(t, dtype=np.int32).reshape(-1)

        kv_rows, base, at = [], {}, 0
        for b in rebuilt:
            n, lo = starts[b] + counts[b], oldest[b]
            # (whole blocks of 32 rows: the padding repeats the last one; the cached row of position j lies at base + j)
            src = slots[b] * cap + np.minimum(np.arange(lo, lo + -(-(n - lo) // 32) * 32, dtype=np.int64), n - 1)
            kv_rows.append(src.astype(np.int32))
            base[b] = at - lo
            at += src.size
        if rebuilt and arena.slots * cap >= 1 << 31:
            raise ValueError("more than 2^31 cached rows in one plane")
        f_rows = others(rebuilt)
        # segments of the matrix memories' prefill
        seg_a = seg_c = chains = np.zeros((0, 4), np.int32)
        seg_end = np.zeros(0, np.int32)
        seg = max(self.SEGMENT, -(-max(counts) // self.MAX_SEGMENTS))
        chunks = self._chunks and seg <= 256
        few = [min(self.SEGMENT, self._few_tokens(len(counts), l.heads, l.dim, l.vdim) if chunks else self.SEGMENT)
               for l in self.config.layers if l.kind == "mlstm"]
        if few and max(counts) > max(few):
            sa, ch = [], []
            for b, (s, s0, c) in enumerate(zip(slots, starts, counts)):
                ch.append((s, s0, len(sa), -(-c // seg)))
                sa += [(len(sa) + k, 0, min(seg, c - q), int(row0[b]) + q) for k, q in enumerate(range(0, c, seg))]
            seg_a = np.asarray(sa, dtype=np.int32)
            seg_c = seg_a.copy()
            seg_c[:, 1] = 1                                 # the second pass starts every segment from a state that was put there
            chains = np.asarray(ch, dtype=np.int32)
            seg_end = np.full(len(sa), -1, dtype=np.int32)  # a request's last segment leaves the slot's new state
            seg_end[chains[:, 2] + chains[:, 3] - 1] = chains[:, 0]
        tables = dict(ids=st.ids, pos=rows[:, 1], want=want_rows, reqs=reqs, s_tiles=rows[others(big)])
        if big:
            tables.update(p_tiles=tiles_of(big, slots))
        if rebuilt:
            # f_: the rows that fold their queries; a_tiles: every row, for layers that fold them all
            tables.update(l_tiles=tiles_of(rebuilt, base), kv_rows=np.concatenate(kv_rows), f_rows=rows[f_rows, 3], a_tiles=rows if self._folds else none)
        if rebuilt != big:
            tables.update(f_tiles=rows[f_rows])
        if self._wide:                             # tiles of 16 queries, for heads too wide for the others
            tables.update(w_tiles=np.asarray([(s, s0 + q, min(16, c - q), int(row0[b]) + q) for b, (s, s0, c) in enumerate(zip(slots, starts, counts))
                                              for q in range(0, c, 16)], dtype=np.int32))
        if seg_end.size:
            tables.update(seg_a=seg_a, seg_c=seg_c, chains=chains, seg_end=seg_end)
        sizes = {k: v.size for k, v in tables.items()}
        n32 = sum(sizes.values())
        o64 = (n32 * 4 + 7) // 8 * 8
        # one block: int32 tables, then int64 cache offsets
        n_off = len(self._sigs) * T
        blob = np.empty(o64 + n_off * 8 + 8, dtype=np.uint8)
        np.concatenate([v.reshape(-1) for v in tables.values()], out=blob[:n32 * 4].view(np.int32))
        offs = blob[o64:o64 + n_off * 8].view(np.int64).reshape(len(self._sigs), T)
        for k, (g, d) in enumerate(self._sigs):
            np.add(st.row_slot * (g * cap * d), st.row_pos * d, out=offs[k])
        dims = dict(T=T, R=R, n_want=int(want_rows.size), n32=n32, o64=o64, sizes=sizes, tile=tile, ones=max(counts) == 1,
                    longest=max((starts[b] + counts[b] for b in {*big, *rebuilt}), default=0),
                    seg=min(seg, max(counts)) if chunks else 0, every=want_rows.size == T and bool((want_rows == np.arange(T)).all()))
        res = self._decode_graphed(arena, blob, dims) if graphed else None
        if res is None:
            dblob = self._upload(blob)
            logits = torch.empty((dims["n_want"], self.V), dtype=torch.float32, device=dev)
            res = self._run(arena, dblob, dims, logits, num_layers, return_streams)
        for s_, c in zip(slots, counts):
            arena.lengths[s_] += c
        if picked is not None:
            res = res[torch.as_tensor(picked, dtype=torch.long, device=dev)] if picked else res[:0]
        return res

    def _tables(self, dblob, d):
        i32 = dblob[:d["n32"] * 4].view(torch.int32)
        sizes = d["sizes"]
        at, out = 0, dict(tile=d["tile"], longest=d["longest"], ones=d["ones"], seg=d["seg"], n_seg=sizes.get("seg_end", 0),
                           n_chains=sizes.get("chains", 0) // 4)
        for name, n in sizes.items():
            out[name] = i32[at:at + n]
            at += n
        for name in ("p_tiles", "l_tiles", "kv_rows", "f_rows", "a_tiles", "w_tiles"):
            out.setdefault(name, i32[:0])
        out.setdefault("f_tiles", out["s_tiles"])  # (the same rows, unless other requests are rebuilt than tiled)
        no = len(self._sigs)
        out["offs"] = dblob[d["o64"]:d["o64"] + no * d["T"] * 8].view(torch.int64).view(no, d["T"])
        return out

    def _run(self, arena, dblob, d, logits, num_layers=None, return_streams=False):
        """The device side of a step: every launch of the forward, reading the step's tables from ``dblob``."""
        dev, E, f32 = self.device, self.dtype, torch.float32
        W, T, R = self.W, d["T"], d["R"]
        tb = self._tables(dblob, d)
        layers = self.layers if num_layers is None else self.layers[:num_layers]
        eps = self.config.norm_eps
        few = T * W <= B.NORM_LINEAR_MAX          # the sizes at which a norm may ride in the launch of the products that read it
        x, spare = self._mat("x", T, W, f32), self._mat("x_next", T, W, f32) if few else None
        h = self._mat("h", T, W, E)
        y1, y2 = self._mat("y1", T, W, f32), self._mat("y2", T, W, f32)
        streams = torch.empty((len(layers), T, W), dtype=f32, device=dev) if return_streams else None
        rows = dict(table=self.embed, ids=tb["ids"], scale=self.config.embed_scale)      # where x comes from, until it is there
        pending = {}                               # the sublayer result that is still to be gated, normed and added to x

        def step(gain, out, **kw):
            nonlocal rows, pending
            if rows:
                B.embed_scaled_rows(*rows.values(), x)
            B.post_norm(x, gain=gain, out=out, eps=eps, n_rows=kw.pop("n_rows", T), **pending, **kw)
            rows, pending = {}, {}

        def project(gain, a, b=None):
            """The products ``a`` and, where given, ``b`` of the normed rows: at few rows (up to eight of 2048 columns) the norm goes into their launch."""
            nonlocal x, spare, rows, pending
            if few and (rows or pending):
                to = x if rows else spare
                if B.norm_linear(a, b, gain, gain if b else None, to, eps=eps, **(rows or dict(x=x, **pending))):
                    x, spare = to, x if to is spare else spare
                    rows, pending = {}, {}
                    return
            if rows:
                B.embed_norm(*rows.values(), x, gain, h, eps=eps)
                rows = {}
            else:
                step(gain, h)
            if b:
                B.linear_pair(a, b)
            else:
                B.linear_run(a)

        # A layer without a feed-forward leaves its residual gate in its projected rows; where the norm that reads it rides in the next layer's projection, that
        # one stores elsewhere.
        mix_in = ("mix_in", "mix_in_next" if few else "mix_in")
        for i, lw in enumerate(layers):
            l = lw["cfg"]
            P = self._mat(mix_in[i % 2], T, lw["w_in"].shape[0], E)
            project(lw["norm1"], B.linear_args(h, lw["w_in"], P, M=T, bias=lw["b_in"], act_split=lw["act_from"], act2=B.ACT_SIGMOID))
            gate, ldg = getattr(self, "_" + l.kind)(arena, i, l, lw, P, y1, tb, T, R)
            pending = dict(y=y1, gate=gate, ldg=ldg, post_gain=lw["norm1b"])
            if l.ff:
                rg = self._mat("ff_gate", T, W, E)
                mid = self._mat("ff_mid", T, l.ff, E)
                project(lw["norm2"], B.linear_args(h, lw["rg2"], rg, M=T, bias=lw["rg2b"], act=B.ACT_SIGMOID),
                        B.linear_args(h, lw["w_gate"], mid, M=T, epilogue=B.EPI_SILU_MUL, w2=lw["w_up"], bias=lw["b_gate"], bias2=lw["b_up"],
                                      act=ACTS[l.act]))
                B.linear(mid, lw["w_down"], y2, M=T, bias=lw["b_down"])
                pending = dict(y=y2, gate=rg, ldg=W, post_gain=lw["norm2b"])
            if streams is not None:
                B.post_norm(x, eps=eps, n_rows=T, x_out=streams[i], **pending)
                pending = {}
        if d["n_want"]:
            nw = d["n_want"]
            hn = self._mat("hn", nw, W, E)
            logit = B.linear_args(hn, self.head, logits, M=nw)
            if few and pending and d["every"] and B.norm_linear(logit, None, self.final_norm, None, spare, eps=eps, x=x, many=True, **pending):
                return (logits, streams) if return_streams else logits
            step(self.final_norm, hn, rows=tb["want"], n_rows=nw)
            B.linear_run(logit)
        return (logits, streams) if return_streams else logits

    # ---- mixers (each gets its projected rows P, leaves its result in y, fp32 [T, W], and returns where the residual gate's sigmoid lies) --------------------
    def _splits(self, n, groups, heads, reach, full=768, unit=64, merged=False):
        """Into how many runs the keys of ``n`` rows are cut (the kernels of single rows: ``n * groups`` workgroups a run, ``full`` of them at a
        time).  Rounds of the chip times a run's blocks of ``unit`` keys and what starting one costs, and the merge, unless that is a launch anyhow (``merged``):
        us, 8 heads over 2, 30 000 keys, cut for 512 workgroups / by this rule: 16 rows 73 / 65, 64 236 / 216, 128 455 / 400, 256 930 / 749, 512 1 678 / 1 381."""
        blocks, w, join = -(-reach // unit), n * groups, 0 if merged else 1 + n * heads / 1200
        best = (-(-w // full) * (blocks + 2), 1)
        if blocks > (1 if merged else 3):
            for k in range(1, 5):
                s = min(64, blocks, full * k // w)
                if s > 1:
                    best = min(best, (-(-w * s // full) * (-(-blocks // s) + 2) + join, s))
        return best[1]

    def _step_splits(self, n, groups, heads, reach, full=768, merged=False):
        """The same for a step's single tokens: in fp32, whose blocks are 32 keys, by these while every block finds a CU of its own.  us a step, width 1024, 64 / 32: one
        of 150 keys 191 / 169, two of 300 183 / 178, of 1000 184 / 180, eight of 300 234 / 229, of 1000 (512 blocks) 234 / 240, 32 of 300 (640) 366 / 368."""
        unit = 32 if self.dtype == torch.float32 and n * groups * -(-reach // 32) <= 256 else 64
        return self._splits(n, groups, heads, reach, full, unit, merged)

    def _latent_step(self, n, groups, reach, splits):
        """Whether a step of ``n`` single tokens goes through ``B.attn_step`` over a latent: it saves a launch, but reads a row twice, as key and as value, where
        ``B.attn_latent`` reads it once.  us, a layer's step, 16 heads over 192 + 64 columns, head_prep and attn_latent / attn_step: bf16 8 of 8 000 keys 59 / 45, 64 of
        2 000 71 / 63, of 8 000 103 / 103, 192 of 2 000 94 / 91, 128 of 4 000 102 / 109, 256 of 4 000 170 / 177, 1 024 of 1 000 219 / 213; fp32 64 of 2 000 118 / 102, 128
        of 4 000 217 / 226, of 8 000 334 / 385, 512 of 1 000 (one run) 255 / 218.  (Heads' own keys: faster at all of 1 .. 1 024 rows, 60 .. 30 000 keys.)"""
        return n * groups * -(-reach // 64) <= 8000 or (splits == 1 and (self.dtype == torch.float32 or n * groups > 768))

    def _attention(self, arena, i, l, lw, P, y, tb, T, R):
        E = self.dtype
        H, G, D, Dv = l.heads, l.kv_heads, l.dim, l.vdim
        HD, GD, GV = H * D, G * D, G * Dv
        N = P.shape[1]
        plane = arena.planes[i]
        vf = self._mat("v_first", T, GV, torch.float32) if l.v_mix else None
        reach = min(arena.cap, l.mask or arena.cap)
        if tb["ones"] and B.attn_step_fits(E, H, G, D, Dv, l.rot_dims):      # (a row's own key is the only new one it sees)
            splits = self._step_splits(T, G * -(-H // (16 * G)), H, reach)
            att, strides = self._mat("mix_out", T, H * Dv, E), (arena.slot_stride(i), arena.head_stride(i), D + Dv)
            part = self._scratch("attn_part", B.attn_softmax_part(T, H, splits, Dv), torch.float32) if splits > 1 else None
            B.attn_step(P, tb["s_tiles"], T, plane, strides, plane.view(-1)[D:], strides, H, G, D, Dv, l.scale, att, q_at=0, q_head_stride=D, k_at=HD,
                        v_at=HD + GD, q_gain=lw["q_gain"], k_gain=lw["k_gain"], eps=self.config.norm_eps, rot_dims=l.rot_dims, freqs=lw["freqs"],
                        rot_mag=lw["rot_mag"], blend=lw["blend"], other=vf if lw["blend"] is not None else None,
                        keep=vf if i == self.first_v_mix else None, block=l.mask, sink=lw["sink"], gate=P[:, HD + GD + GV:], ldg=N, n_splits=splits, part=part)
            B.linear(att, lw["wo"], y, M=T)
            return P[:, HD + GD + GV + H:], N
        q = self._mat("q_rows", T, HD, E)
        row = dict(row_off=tb["offs"][self._sigs.index((G, D + Dv))], head_stride=arena.head_stride(i))
        segs = [B.head_seg(P, N, H, D, q, norm=True, gain=lw["q_gain"], rot_dims=l.rot_dims, ld_dst=HD),
                B.head_seg(P[:, HD:], N, G, D, plane, norm=True, gain=lw["k_gain"], rot_dims=l.rot_dims, **row),
                B.head_seg(P[:, HD + GD:], N, G, Dv, plane, norm=True, blend=lw["blend"], other=vf if lw["blend"] is not None else None,
                           keep=vf if i == self.first_v_mix else None, dst_offset=D, **row)]
        B.head_prep(segs, T, E, pos=tb["pos"], freqs=lw["freqs"], rot_mag=lw["rot_mag"], eps=self.config.norm_eps)
        att = self._mat("mix_out", T, H * Dv, E)
        values, gate = plane.view(-1)[D:], P[:, HD + GD + GV:]
        ss, hs, rs = arena.slot_stride(i), arena.head_stride(i), D + Dv
        if D > 256:
            n = tb["w_tiles"].numel() // 4
            splits = 1 if n * H >= 512 or arena.cap <= 256 else max(1, min(16, 1024 // (n * H), arena.cap // 128))
            part = self._scratch("attn_part", B.attn_softmax_part(T, H, splits, Dv), torch.float32) if splits > 1 else None
            B.attn_softmax(q, HD, tb["w_tiles"], n, plane, (ss, hs, rs), plane, D, (ss, hs, rs), False, H, G, D, Dv, l.scale, att,
                           block=l.mask, sink=lw["sink"], gate=gate, ldg=N, gate_per_head=True, n_splits=splits, part=part)
        else:
            kw = dict(ldo=H * Dv, block=l.mask, sink=lw["sink"], gate=gate, ldg=N)
            n = tb["p_tiles"].numel() // 4
            if n:
                B.attn_prompt(q, tb["p_tiles"], n, tb["tile"], plane, (rs, hs, ss), values, (rs, hs, ss), H, G, D, Dv, l.scale, att,
                              longest=tb["longest"], **kw)
            n = tb["s_tiles"].numel() // 4
            if n:
                splits = self._splits(n, G * -(-H // (16 * G)), H, reach, 768 if max(D, Dv) <= 128 else 512)
                part = self._scratch("attn_part", B.attn_softmax_part(n, H, splits, Dv), torch.float32) if splits > 1 else None
                B.attn_rows(q, tb["s_tiles"], n, plane, (ss, hs, rs), values, (ss, hs, rs), H, G, D, Dv, l.scale, att, gate_per_head=True,
                            n_splits=splits, part=part, **kw)
        B.linear(att, lw["wo"], y, M=T)
        return P[:, HD + GD + GV + H:], N

    def _latent_attention(self, arena, i, l, lw, P, y, tb, T, R):
        E = self.dtype
        H, D, Rd, Dv, C = l.heads, l.dim, l.rot_dim, l.vdim, l.kv_rank
        DR, HQ, HV, CR = D + Rd, H * (D + Rd), H * Dv, C + Rd
        N = P.shape[1]
        plane = arena.planes[i]
        off = tb["offs"][self._sigs.index((1, CR))]
        tiled = lw["prompts"] and tb["l_tiles"].numel() > 0
        f_tiles = tb["f_tiles"] if lw["prompts"] or not tb["a_tiles"].numel() else tb["a_tiles"]
        n = f_tiles.numel() // 4
        qa = self._mat("q_latent", T, H * CR, E) if n else None   # per head [W_uk^T q | rotated part]: a query over the cached rows
        reach = min(arena.cap, l.mask or arena.cap)
        full = 768 if CR <= 256 else 512
        # the heads' up-projections and gates ride in the launch that merges: us a step of 16 heads, bf16, without / with it: one of 300 keys 212 / 206, 8 of 300
        # 287 / 281, 32 of 100 360 / 356, 64 of 60 397 / 396; 8 heads, fp32, two of 300 189 / 183
        up = T <= 64 and Dv <= 128 and Dv % 8 == 0
        one = tb["ones"] and n == T and B.attn_step_fits(E, H, 1, CR, C, Rd, True)
        splits = self._step_splits(T, -(-H // 16), H, reach, full, up) if one else 0
        if one and self._latent_step(T, -(-H // 16), reach, splits):
            B.linear(P, lw["w_abs"], qa, M=T, n_batch=H, ldx=N, x_batch_stride=DR, ldy=H * CR, y_batch_stride=CR)
            strides, og, gate = (arena.slot_stride(i), 0, CR), self._mat("mix_gated", T, HV, E), P[:, HQ + CR:]
            kw = dict(q_at=D, q_head_stride=DR, k_at=HQ, q=qa, k_gain=lw["c_gain"], eps=self.config.norm_eps, rot_dims=Rd, freqs=lw["freqs"],
                      rot_mag=lw["rot_mag"], window=l.mask, n_splits=splits)
            part = self._scratch("attn_part", B.attn_softmax_part(n, H, splits, C), torch.float32)
            if up:
                B.attn_step(P, f_tiles, T, plane, strides, plane, strides, H, 1, CR, C, l.scale, og, part=part, up=lw["w_uv"], up_gate=gate, ld_up_gate=N, **kw)
            else:
                ol, ov = self._mat("mix_out", T, H * C, E), self._mat("mix_o32", T, HV, torch.float32)
                B.attn_step(P, f_tiles, T, plane, strides, plane, strides, H, 1, CR, C, l.scale, ol, part=part, **kw)
                B.linear(ol, lw["w_uv"], ov, M=T, n_batch=H, ldx=H * C, x_batch_stride=C, ldy=HV, y_batch_stride=Dv)
                B.gated_norm(ov, None, gate, N, og, self.config.norm_eps, T)
            B.linear(og, lw["wo"], y, M=T)
            return P[:, HQ + CR + HV:], N
        splits = self._splits(n, -(-H // 16), H, reach, full) if n else 0
        q = self._mat("q_rows", T, HQ, E) if tiled else None      # per head [plain part | rotated part]: a query over rebuilt rows
        segs = [B.head_seg(P[:, HQ:], N, 1, C, plane, norm=True, gain=lw["c_gain"], row_off=off)]
        if tiled:
            segs.append(B.head_seg(P, N, H, D, q, src_head_stride=DR, ld_dst=HQ, head_stride=DR))
        if Rd:
            segs.append(B.head_seg(P[:, HQ + C:], N, 1, Rd, plane, rot_dims=Rd, row_off=off, dst_offset=C))
            if tiled:
                segs.append(B.head_seg(P[:, D:], N, H, Rd, q, src_head_stride=DR, rot_dims=Rd, ld_dst=HQ, head_stride=DR, dst_offset=D))
            if n:
                segs.append(B.head_seg(P[:, D:], N, H, Rd, qa, src_head_stride=DR, rot_dims=Rd, ld_dst=H * CR, head_stride=CR, dst_offset=C))
        for k in range(0, len(segs), 4):
            B.head_prep(segs[k:k + 4], T, E, pos=tb["pos"], freqs=lw["freqs"], rot_mag=lw["rot_mag"], eps=self.config.norm_eps)
        og, gate = self._mat("mix_gated", T, HV, E), P[:, HQ + CR:]
        if n:
            rows = tb["f_rows"] if tiled and n < T else None
            B.linear(P, lw["w_abs"], qa, M=n, row_src=rows, row_dst=rows, n_batch=H, ldx=N, x_batch_stride=DR, ldy=H * CR, y_batch_stride=CR)
            ol = self._mat("mix_out", T, H * C, E)
            part = self._scratch("attn_part", B.attn_softmax_part(n, H, splits, C), torch.float32) if splits > 1 else None
            B.attn_latent(qa, f_tiles, n, plane, arena.slot_stride(i), CR, H, CR, C, l.scale, ol, window=l.mask, n_splits=splits, part=part)
            ov = self._mat("mix_o32", T, HV, torch.float32)
            B.linear(ol, lw["w_uv"], ov, M=n, row_src=rows, row_dst=rows, n_batch=H, ldx=H * C, x_batch_stride=C, ldy=HV, y_batch_stride=Dv)
            B.gated_norm(ov, None, gate, N, og, self.config.norm_eps, T)
        if tiled:
            # (after the others: their gate runs over all rows)
            flat, M, ew = plane.view(-1, CR), tb["kv_rows"].numel(), D + Dv
            Hs = max(1, min(H, self.REBUILD_BYTES // (M * ew * plane.element_size())))
            kv = self._mat("kv_rows", M, Hs * ew, E)
            for h0 in range(0, H, Hs):
                n_h = min(Hs, H - h0)
                if n_h == H:
                    B.linear(flat, lw["w_kv"], kv, M=M, row_src=tb["kv_rows"], ldx=CR)
                else:
                    for at, w in ((0, lw["w_kv"][h0 * D:(h0 + n_h) * D]), (n_h * D, lw["w_kv"][H * D + h0 * Dv:H * D + (h0 + n_h) * Dv])):
                        B.linear(flat, w, kv[:, at:], M=M, row_src=tb["kv_rows"], ldx=CR, ldy=Hs * ew)
                qh, oh, gh = (q, og, gate) if not h0 else (q[:, h0 * DR:], og[:, h0 * Dv:], gate[:, h0 * Dv:])
                B.attn_prompt(qh, tb["l_tiles"], tb["l_tiles"].numel() // 4, tb["tile"], kv, (Hs * ew, D), kv[:, n_h * D:], (Hs * ew, Dv),
                              n_h, n_h, DR, Dv, l.scale, oh, ldq=HQ, ldo=HV, k_tail=flat[:, C:] if Rd else None, tail_row_stride=CR,
                              tail_rows=tb["kv_rows"], tail_dim=Rd, window=l.mask, gate=gh, ldg=N, gate_cols=True, longest=tb["longest"])
        B.linear(og, lw["wo"], y, M=T)
        return P[:, HQ + CR + HV:], N

    def _mlstm(self, arena, i, l, lw, P, y, tb, T, R):
        H, D, Dv = l.heads, l.dim, l.vdim
        HD, HV = H * D, H * Dv
        N = P.shape[1]
        cols = (P, P[:, HD:], P[:, 2 * HD:], P[:, 2 * HD + HV:], P[:, 2 * HD + HV + H:], N)
        state, ns = arena.states[i][0], tb["n_seg"]
        rec = B.mlstm_state_floats(H, D, Dv)
        local, start, fsum = (self._mat("seg_local", ns, rec, torch.float32), self._mat("seg_start", ns, rec, torch.float32),
                              self._mat("seg_logf", ns, H, torch.float32)) if ns else (None, None, None)
        gate, on = P[:, 2 * HD + HV + 2 * H:], self._mat("mix_gated", T, HV, self.dtype)
        tail = (H, D, Dv, D ** -0.5, l.gate_cap)
        if ns and tb["seg"]:
            B.mlstm_prompt(cols[:5], N, tb["seg_a"], ns, tb["chains"], tb["n_chains"], tb["seg"], tb["seg_end"], state, *tail, lw["gain"], gate, N, on,
                           self.config.norm_eps, local, fsum, start)
        elif tb["ones"] and B.mlstm_step_fits(D, Dv, N, cols[2]):
            B.mlstm_step(cols[:5], N, tb["reqs"], R, state, *tail, lw["gain"], gate, N, on, self.config.norm_eps)
        else:
            o = self._mat("mix_o32", T, HV, torch.float32)
            if ns:
                # every segment from nothing (only the states move), the segments chained, then every segment from its start state
                B.mlstm(*cols, tb["seg_a"], ns, local, *tail, None, from_nothing=True, log_f_sum=fsum)
                B.mlstm_chain(local, fsum, start, state, tb["chains"], tb["n_chains"], H, D, Dv)
                B.mlstm(*cols, tb["seg_c"], ns, start, *tail, o, end_slots=tb["seg_end"], end_state=state)
            else:
                B.mlstm(*cols, tb["reqs"], R, state, *tail, o)
            B.gated_norm(o, lw["gain"], gate, N, on, self.config.norm_eps, T, group=Dv)
        B.linear(on, lw["wo"], y, M=T)
        return P[:, 2 * HD + 2 * HV + 2 * H:], N
