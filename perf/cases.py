"""What a user of this package has it do, as measurable cases.

Two kinds of programs use the package, and the cases come from both:

* the prompt cache proper (``CacheEngine`` over a Llama-2 / CodeLlama / MPT adapter): a schema is encoded once (``encode``), prompts
  are answered over its staged module KV (``question``), tokens are decoded behind them (``decode``), and the same prompt is run
  without the cache (``prompt``).  Layer sizes are those of Llama-2-7b / 13b, CodeLlama-7b and MPT-7b; where a case keeps fewer layers
  than the model has, every layer is alike and the rest would repeat it.
* serving requests in batches (``BatchEngine.step``) with the designs of the building-block library (``serve``): prompts are
  prefilled together, then every request decodes one token per step.  Kazolorn (talking heads, keys as values, a window,
  polynomial feed-forwards) and Fivesun (softmax, latent and matrix-memory mixers) at the sizes ``bench.py`` runs them.  Feed-forwards
  are dense: with routed experts a rounding difference picks another expert, and outputs could not be compared.

(``load_in_8bit`` is left out for the same reason: its activation codes turn a relative difference of 1e-7 at the input of one layer
into 1e-2 at the logits.)

Weights, tokens and texts are drawn from the seed; there are no checkpoints here.  Next tokens are given, not sampled, so that a pass
computes the same thing whatever the rounding.
"""
import math
import os
import re
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "prompt-cache_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

DEV = "cuda:0"
SIZES = {  # width, feed-forward, heads, rotary base (heads have 128 columns everywhere)
    "llama2-7b": (4096, 11008, 32, 10000.0),
    "codellama-7b": (4096, 11008, 32, 1000000.0),
    "llama2-13b": (5120, 13824, 40, 10000.0),
    "mpt-7b": (4096, 16384, 32, 0.0),
}
VOCAB = 32000


# ---- the cases ------------------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # the headline: a persona prompt of ~1.7 k cached tokens in six picked union members and a short question, all 32 layers
        dict(name="question 7b persona", kind="question", model="llama2-7b", layers=32, text=376, docs=0, doc_len=0, unions=6,
             members=2, member_len=224, question=12),
        # reading comprehension over one cached passage: a few hundred tokens, a question of two row tiles
        dict(name="question 7b passage", kind="question", model="codellama-7b", layers=16, text=21, docs=1, doc_len=287, unions=0,
             members=0, member_len=0, question=27),
        # long context: one document of 8 k tokens, a question of ~260 tokens, 13b layers
        dict(name="question 13b long document", kind="question", model="llama2-13b", layers=8, text=11, docs=1, doc_len=8247, unions=0,
             members=0, member_len=0, question=259),
        # the other position scheme of the reference's adapters (ALiBi over full position ids)
        dict(name="question mpt", kind="question", model="mpt-7b", layers=8, text=33, docs=3, doc_len=301, unions=0, members=0,
             member_len=0, question=19),
        # generation behind a cached prompt: eight tokens, one lm() call each
        dict(name="decode 7b", kind="decode", model="llama2-7b", layers=32, text=376, docs=2, doc_len=675, unions=0, members=0,
             member_len=0, question=12, tokens=8),
        # a schema is added: one trunk and its union members, the package's bulk work
        dict(name="encode 7b schema", kind="encode", model="llama2-7b", layers=8, text=376, docs=0, doc_len=0, unions=6, members=5,
             member_len=224, question=12),
        # the same prompt without the cache, every token through the model
        dict(name="prompt 7b no cache", kind="prompt", model="llama2-7b", layers=8, text=376, docs=2, doc_len=675, unions=0, members=0,
             member_len=0, question=11),
        # one long prompt through each of the two served designs
        dict(name="serve kazolorn prompt", kind="serve", model="kazolorn", width=2048, requests=1, prompt=2048, tokens=0, dtype="bf16"),
        dict(name="serve fivesun prompt", kind="serve", model="fivesun", width=2048, requests=1, prompt=2048, tokens=0, dtype="bf16"),
        # eight requests that decode together
        dict(name="serve fivesun batch", kind="serve", model="fivesun", width=2048, requests=8, prompt=300, tokens=16, dtype="bf16"),
        # the design's 32-bit mode
        dict(name="serve fivesun f32", kind="serve", model="fivesun", width=1024, requests=2, prompt=300, tokens=8, dtype="f32"),
        # the smallest: a lone request, a short prompt, a narrow model, mostly launch latency
        dict(name="serve kazolorn lone", kind="serve", model="kazolorn", width=1024, requests=1, prompt=37, tokens=8, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    if rng.random() < 0.6:
        kind = rng.choice(["question", "question", "question", "decode", "encode", "prompt"])
        model = rng.choice(["llama2-7b", "codellama-7b", "llama2-13b", "mpt-7b"])
        c = dict(kind=kind, model=model, layers=rng.randint(4, 8), text=_log(rng, 8, 500), docs=0, doc_len=0, unions=0, members=0,
                 member_len=0, question=_log(rng, 1, 300))
        if kind == "encode" or (kind == "question" and rng.random() < 0.4):
            c.update(text=_log(rng, 64, 500), unions=rng.randint(1, 6), members=rng.randint(2, 4), member_len=_log(rng, 40, 260))
        else:
            c.update(docs=rng.randint(1, 4), doc_len=_log(rng, 60, 900))
        if kind == "decode":
            c.update(tokens=rng.randint(2, 8))
        return c
    model = rng.choice(["kazolorn", "fivesun"])
    c = dict(kind="serve", model=model, width=rng.choice([512, 1024, 2048]), requests=_log(rng, 1, 8), prompt=0, tokens=0,
             dtype=rng.choice(["bf16", "bf16", "bf16", "f32"]))
    if rng.random() < 0.5:
        c.update(prompt=_log(rng, 100, 2048 // c["requests"]))
    else:
        c.update(prompt=_log(rng, 9, 300), tokens=rng.randint(4, 16))
    return c


# ---- the schema of a prompt-cache case ---------------------------------------------------------------------------------------------------
class Words:
    """A tokenizer of whole words: ``w17`` with the white space in front of it is token 4 + 17, white space alone token 3."""
    unk_token, unk_token_id, bos_token_id, eos_token, eos_token_id = "<unk>", 0, 1, "</s>", 2

    def encode(self, text, add_special_tokens=False):
        return [3 if p.isspace() else 4 + int(p.strip()[1:]) for p in re.findall(r"\s*\S+|\s+", text)]

    def decode(self, ids, **_):
        return " ".join("w%d" % (i - 4) for i in ids)


def _schema(case, seed):
    """(schema text, prompt text, trunk, members, question): the texts for the engine; ``trunk`` = the (token, position) pairs outside
    all unions, in order; ``members`` = per picked union member the length of the trunk in front of it and its own pairs."""
    g = torch.Generator().manual_seed(seed * 31 + 7)

    def words(n):
        return torch.randint(0, VOCAB - 4, (n,), generator=g).tolist()

    def text(ws):
        return " ".join("w%d" % w for w in ws)

    trunk, picked, refs, pos = [], [], [], 0

    def put(ws):
        nonlocal pos
        trunk.extend((4 + w, pos + i) for i, w in enumerate(ws))
        pos += len(ws)

    ws = words(case["text"])
    out = ['<schema name="s">', text(ws)]
    put(ws)
    for d in range(case["docs"]):
        ws = words(case["doc_len"])
        out.append('<module name="d%d">%s</module>' % (d, text(ws)))
        refs.append("<d%d/>" % d)
        put(ws)
    for u in range(case["unions"]):
        pick, start, longest = (u + 1) % case["members"], pos, 0
        out.append('<module name="u%d"><union>' % u)
        for m in range(case["members"]):
            n = max(1, case["member_len"] - 7 * ((3 * m + u) % 4))
            longest = max(longest, n)
            ws = words(n)
            out.append('<module name="u%d-%d">%s</module>' % (u, m, text(ws)))
            if m == pick:
                picked.append((len(trunk), [(4 + w, start + i) for i, w in enumerate(ws)]))
        refs.append("<u%d><u%d-%d/></u%d>" % (u, u, pick, u))
        out.append("</union></module>\n")
        pos = start + longest
        trunk.append((3, pos))
        pos += 1
    out.append("</schema>")
    ws = words(case["question"])
    question = [(4 + w, pos + i) for i, w in enumerate(ws)]
    prompt = '<prompt schema="s">%s%s</prompt>' % ("".join(refs), " ".join("w%d" % w for w in ws))
    return "".join(out), prompt, trunk, picked, question


def _staged(case):
    """Cached tokens of the prompt, and tokens that an encode of the schema runs (each once)."""
    members = [max(1, case["member_len"] - 7 * ((3 * m + u) % 4)) for u in range(case["unions"]) for m in range(case["members"])]
    picked = [max(1, case["member_len"] - 7 * ((3 * ((u + 1) % case["members"]) + u) % 4)) for u in range(case["unions"])]
    trunk = case["text"] + case["docs"] * case["doc_len"] + case["unions"]
    return trunk + sum(picked), trunk + sum(members)


# ---- weights -----------------------------------------------------------------------------------------------------------------------------
def _draw_tensors(shapes, seed, dtype):
    """name -> (shape, mean, deviation) drawn on the device, in the order given."""
    g = torch.Generator(device=DEV).manual_seed(seed * 977 + 13)
    return {k: torch.randn(shp, generator=g, device=DEV, dtype=dtype).mul_(sd).add_(mean) if mean else
            torch.randn(shp, generator=g, device=DEV, dtype=dtype).mul_(sd) for k, (shp, mean, sd) in shapes.items()}


def _decoder_weights(case, seed):
    """fp16 weights of the Llama and MPT adapters: N(0, 0.02) matrices, gains around 1."""
    w, ff, _, _ = SIZES[case["model"]]
    s, mat, gain = {}, (lambda *shp: (shp, 0.0, 0.02)), ((w,), 1.0, 0.1)
    s["embed"] = mat(VOCAB, w)
    for i in range(case["layers"]):
        p = "l%d." % i
        s[p + "ln1"], s[p + "ln2"] = gain, gain
        if case["model"].startswith("mpt"):
            s[p + "wqkv"], s[p + "wo"], s[p + "w1"], s[p + "w2"] = mat(3 * w, w), mat(w, w), mat(ff, w), mat(w, ff)
        else:
            s[p + "wq"], s[p + "wk"], s[p + "wv"], s[p + "wo"] = mat(w, w), mat(w, w), mat(w, w), mat(w, w)
            s[p + "gate"], s[p + "up"], s[p + "down"] = mat(ff, w), mat(ff, w), mat(w, ff)
    s["lnf" if case["model"].startswith("mpt") else "norm"] = gain
    s["lm_head"] = mat(VOCAB, w)
    return _draw_tensors(s, seed, torch.float16)


def _served_shape(case):
    from promptcache_amd.model.config import FivesunShape, KazolornShape
    w = case["width"]
    h = w // 128
    if case["model"] == "kazolorn":
        return KazolornShape.uniform(VOCAB, w, 4, h, h // 4, 128, 1024, 4 * w)
    return FivesunShape.uniform(VOCAB, w, ["attention", "latent_attention", "attention", "mlstm"], h, h // 4, 128, 2 * w, chunk=1024,
                                window=1024, kv_rank=192, rot_dim=64)


def _served_weights(case, seed):
    """bfloat16 weights of the served designs: matrices scaled by their depth, gains and layer scales around 1 and 0.5, biases that
    are not zero, depth weights that favour the newest result, forget gates that keep the memory for tens of tokens."""
    w, h, d, ff = case["width"], case["width"] // 128, 128, (4 if case["model"] == "kazolorn" else 2) * case["width"]
    kv, rank, rot = h // 4, 192, 64
    s, mat, gain, bias = {}, (lambda n, k: ((n, k), 0.0, k ** -0.5)), (lambda n: ((n,), 1.0, 0.1)), (lambda n: ((n,), 0.0, 0.1))
    s["embed"] = ((VOCAB, w), 0.0, 1.0 if case["model"] == "kazolorn" else w ** -0.5)
    for i in range(4):
        p, m = "l%d." % i, "l%d.mix." % i
        if case["model"] == "kazolorn":
            s[p + "norm1"], s[p + "norm2"], s[p + "ls1"], s[p + "ls2"] = gain(w), gain(w), ((w,), 0.5, 0.1), ((w,), 0.5, 0.1)
            s[m + "q"], s[m + "q.b"], s[m + "k"], s[m + "k.b"] = mat(h * d, w), bias(h * d), mat(kv * d, w), bias(kv * d)
            s[m + "o"], s[m + "o.b"], s[m + "talk"] = mat(w, h * d), bias(w), ((h, h), 0.0, 0.2)
            s[p + "mlp.up"], s[p + "mlp.down"], s[p + "mlp.act"] = mat(ff, w), mat(w, ff), ((4,), 0.4, 0.2)
            s[p + "dwa"] = ((i + 2,), 0.0, 0.15)
            continue
        s[p + "norm1"], s[p + "norm1b"], s[p + "rg1"], s[p + "rg1.b"] = gain(w), gain(w), mat(w, w), bias(w)
        if i in (0, 2):
            s[m + "q"], s[m + "k"], s[m + "v"] = mat(h * d, w), mat(kv * d, w), mat(kv * d, w)
            s[m + "q.norm"], s[m + "k.norm"], s[m + "sink"] = gain(d), gain(d), ((h,), 0.0, 0.8)
            s[m + "g"], s[m + "o"], s[m + "vmix"] = mat(h, w), mat(w, h * d), ((1,), 0.35, 0.1)
        elif i == 1:
            s[m + "q"], s[m + "dkv"], s[m + "dkv.norm"] = mat(h * (d + rot), w), mat(rank + rot, w), gain(rank)
            s[m + "uk"], s[m + "uv"], s[m + "g"], s[m + "o"] = mat(h * d, rank), mat(h * d, rank), mat(h * d, w), mat(w, h * d)
        else:
            s[m + "q"], s[m + "k"], s[m + "v"], s[m + "g"], s[m + "o"] = (mat(w, w) for _ in range(5))
            s[m + "i"], s[m + "i.b"], s[m + "f"], s[m + "f.b"], s[m + "norm"] = mat(h, w), bias(h), mat(h, w), ((h,), 3.0, 0.5), gain(h * d)
        s[p + "norm2"], s[p + "norm2b"], s[p + "rg2"], s[p + "rg2.b"] = gain(w), gain(w), mat(w, w), bias(w)
        for nm, (n, k) in (("gate", (ff, w)), ("up", (ff, w)), ("down", (w, ff))):
            s[p + "mlp." + nm], s[p + "mlp." + nm + ".b"] = mat(n, k), bias(n)
    s["final.norm"], s["head"] = gain(w), mat(VOCAB, w)
    t = _draw_tensors(s, seed, torch.bfloat16)
    for k in t:
        if k.endswith("talk"):
            t[k] += torch.eye(h, device=DEV, dtype=torch.bfloat16)
        elif k.endswith("dwa"):
            t[k][-1] += 1.0
        elif k.endswith("vmix"):
            t[k] = t[k].reshape(())
    return t


def _requests(case, seed):
    g = torch.Generator().manual_seed(seed * 53 + 3)
    return torch.randint(0, VOCAB, (case["requests"], case["prompt"] + case["tokens"]), generator=g).tolist()


# ---- a pass ------------------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    if case["kind"] == "serve":
        from promptcache_amd import BatchEngine
        from promptcache_amd.model import Fivesun, Kazolorn
        cls = Kazolorn if case["model"] == "kazolorn" else Fivesun
        lm = cls(shape=_served_shape(case), weights=_served_weights(case, seed), tokenizer=Words(), device=DEV,
                 dtype=torch.bfloat16 if case["dtype"] == "bf16" else torch.float32)
        n, p = case["requests"], case["prompt"]
        toks = _requests(case, seed)
        steps = [[(r, toks[r][:p], [p - 1]) for r in range(n)]] + \
                [[(r, [toks[r][p + t]], [0]) for r in range(n)] for t in range(case["tokens"])]
        return dict(case=case, engine=BatchEngine(lm, max_tokens=p + case["tokens"]), steps=steps)
    from promptcache_amd import CacheEngine, Prompt
    from promptcache_amd.model import CodeLlama, Llama2, Mpt
    from promptcache_amd.model.config import LlamaShape, MptShape
    w, ff, heads, theta = SIZES[case["model"]]
    weights = _decoder_weights(case, seed)
    if case["model"].startswith("mpt"):
        lm = Mpt(shape=MptShape(vocab_size=VOCAB, hidden_size=w, num_hidden_layers=case["layers"], num_attention_heads=heads),
                 weights=weights, tokenizer=Words(), device=DEV)
    else:
        shape = LlamaShape(vocab_size=VOCAB, hidden_size=w, intermediate_size=ff, num_hidden_layers=case["layers"],
                           num_attention_heads=heads, num_key_value_heads=heads, rope_theta=theta)
        lm = (CodeLlama if case["model"].startswith("code") else Llama2)(shape=shape, weights=weights, tokenizer=Words(), device=DEV)
    del weights
    schema, prompt, _, _, question = _schema(case, seed)
    room = question[-1][1] + 64
    state = dict(case=case, lm=lm, schema=schema, room=room, prompt=Prompt(prompt))
    if case["kind"] == "encode":
        return state
    engine = state["engine"] = CacheEngine(room, lm)
    engine.add_schema(schema)
    if case["kind"] == "decode":
        ids, pos, _, cache = engine.process(state["prompt"], return_full_position_ids=lm.use_full_position_ids)
        out = lm(input_ids=torch.tensor([ids]), position_ids=torch.tensor([pos]), past_key_values=cache, use_cache=True)
        g = torch.Generator().manual_seed(seed * 53 + 3)
        state.update(past=out.past_key_values, positions=list(pos), next=torch.randint(4, VOCAB, (case["tokens"],), generator=g).tolist())
    return state


def run(state):
    case = state["case"]
    if case["kind"] == "serve":
        engine, steps = state["engine"], state["steps"]
        logits = [engine.step(s, end=range(case["requests"]) if i == len(steps) - 1 else ()) for i, s in enumerate(steps)]
        return logits
    lm = state["lm"]
    if case["kind"] == "encode":
        from promptcache_amd import CacheEngine
        engine = CacheEngine(state["room"], lm)
        engine.add_schema(state["schema"])
        segments = sorted(engine.schemas["s"].cache_l1.values(), key=lambda s: (s.token_sequence.offset, len(s), s.token_sequence.text))
        return [s.store for s in segments]
    if case["kind"] == "decode":
        past, pos, logits = state["past"], list(state["positions"]), []
        for t in state["next"]:
            at = pos[-1] + 1
            pos = pos + [at] if lm.use_full_position_ids else [at]
            out = lm(input_ids=torch.tensor([[t]]), position_ids=torch.tensor([pos]), past_key_values=past, use_cache=True)
            past = out.past_key_values
            logits.append(out.logits)
        return logits
    engine = state["engine"]
    engine.prompt_cache.reset()           # another prompt stood there before: every staged row is gathered
    ids, pos, _, cache = engine.process(state["prompt"], no_cache=case["kind"] == "prompt",
                                        return_full_position_ids=lm.use_full_position_ids)
    return lm(input_ids=torch.tensor([list(ids)]), position_ids=torch.tensor([list(pos)]), past_key_values=cache, use_cache=True).logits


# ---- what a pass cannot do without -------------------------------------------------------------------------------------------------------
def work(case):
    if case["kind"] == "serve":
        w, n, p, t = case["width"], case["requests"], case["prompt"], case["tokens"]
        h, kv, es = w // 128, w // 512, 2 if case["dtype"] == "bf16" else 4
        if case["model"] == "kazolorn":
            per, row = 4 * (2 * w * w + kv * 128 * w + 8 * w * w), 4 * kv * 128
            pair = 4 * 4 * w + 4 * 2 * h * h
        else:
            per = 4 * (w * w + 7 * w * w) + 2 * (2 * w * w + 2 * kv * 128 * w) + \
                (h * 192 * w + 256 * w + 2 * h * 128 * 192 + 2 * w * w) + 5 * w * w
            row, pair = 2 * 2 * kv * 128 + 256, (2 * 4 + 5) * w
        seen = sum(min(i + 1, 1024) for i in range(p))
        flops = n * ((p + t) * 2 * per + (1 + t) * 2 * VOCAB * w + pair * (seen + t * min(p, 1024)))
        nbytes = (1 + t) * es * (per + VOCAB * w) + n * es * row * (p + t + t * min(p, 1024)) + (1 + t) * n * VOCAB * 4
        return {"bytes": nbytes, "flops": flops}
    w, ff, _, _ = SIZES[case["model"]]
    L = case["layers"]
    per, head, kv = L * (4 * w * w + (2 if case["model"].startswith("mpt") else 3) * w * ff), VOCAB * w, 4 * L * w
    staged, encoded = _staged(case)
    q = case["question"]
    if case["kind"] == "question":
        return {"bytes": 2 * per + 2 * head + kv * (staged + q) + 4 * q * VOCAB,
                "flops": 2 * q * (per + head) + 4 * L * w * q * (staged + q / 2)}
    if case["kind"] == "decode":
        t = case["tokens"]
        return {"bytes": t * (2 * per + 2 * head + kv * (staged + q + t / 2) + 4 * VOCAB),
                "flops": t * (2 * (per + head) + 4 * L * w * (staged + q))}
    if case["kind"] == "prompt":
        n = staged + q
        return {"bytes": 2 * per + 2 * head + kv * n + 4 * n * VOCAB, "flops": 2 * n * (per + head) + 2 * L * w * n * n}
    pairs = staged * case["text"] / 2 + encoded * case["text"] if case["unions"] else staged * staged / 2
    return {"bytes": 2 * per + kv * encoded, "flops": 2 * encoded * per + 4 * L * w * pairs}


def tolerance(case):
    """fp16 K / V rows and bf16 activations decide: measured against ``exact`` and between summation orders, times four."""
    if case["kind"] == "serve":
        return {"rel": 1e-5, "max": 1e-3} if case["dtype"] == "f32" else {"rel": 0.03, "max": 0.3}
    return {"rel": 1e-2, "max": 0.1}


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------------------
def _f(t):
    return t.to(torch.float64)


def _rms(x, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps)


def _decoder(case, wt, tokens, positions, past, key_positions=None):
    """One call of a Llama or MPT decoder: (logits-to-be [n, width], [(K, V)] of the new rows).  ``past``: per layer (K, V) [m, H, 128];
    every new row sees them and the new rows up to itself."""
    w, ff, H, theta = SIZES[case["model"]]
    mpt = case["model"].startswith("mpt")
    n = len(tokens)
    pos = torch.tensor(positions, device=DEV, dtype=torch.float64)
    m = 0 if past is None else past[0][0].shape[0]
    x = _f(wt["embed"][torch.tensor(tokens, device=DEV)])

    def lin(a, b):
        return a @ _f(b).T

    if mpt:
        kpos = torch.tensor(key_positions, device=DEV, dtype=torch.float64)
        slopes = [2.0 ** (-8.0 * (h + 1) / H) for h in range(H)]

        def norm(v, g):
            v = v - v.mean(-1, keepdim=True)
            return _rms(v, 1e-5) * _f(g)
    else:
        ang = pos[:, None] * theta ** (-torch.arange(0, 128, 2, device=DEV, dtype=torch.float64) / 128)
        cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

        def norm(v, g):
            return _rms(v, 1e-5) * _f(g)

        def turn(v):
            a, b = v[..., :64], v[..., 64:]
            return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
    hidden = torch.ones(n, n, device=DEV, dtype=torch.bool).triu(1)
    kv = []
    for i in range(case["layers"]):
        p = "l%d." % i
        h = norm(x, wt[p + "ln1"])
        if mpt:
            q, k, v = (t.view(n, H, 128) for t in lin(h, wt[p + "wqkv"]).split(w, 1))
        else:
            q, k, v = (t.view(n, H, 128) for t in lin(h, torch.cat([wt[p + "wq"], wt[p + "wk"], wt[p + "wv"]])).split(w, 1))
            q, k = turn(q), turn(k)
        kv.append((k, v))
        if m:
            k, v = torch.cat([past[i][0], k]), torch.cat([past[i][1], v])
        att = torch.empty(n, H, 128, device=DEV, dtype=torch.float64)
        for hd in range(H):
            s = (q[:, hd] @ k[:, hd].T) * 128 ** -0.5
            if mpt:
                s += slopes[hd] * kpos
            s[:, m:].masked_fill_(hidden, -math.inf)
            att[:, hd] = torch.softmax(s, -1) @ v[:, hd]
        x = x + lin(att.reshape(n, w), wt[p + "wo"])
        h = norm(x, wt[p + "ln2"])
        if mpt:
            x = x + lin(torch.nn.functional.gelu(lin(h, wt[p + "w1"])), wt[p + "w2"])
        else:
            gu = lin(h, torch.cat([wt[p + "gate"], wt[p + "up"]]))
            x = x + lin(torch.nn.functional.silu(gu[:, :ff]) * gu[:, ff:], wt[p + "down"])
    return norm(x, wt["lnf" if mpt else "norm"]), kv


def _exact_decoder(case, seed):
    wt = _decoder_weights(case, seed)
    _, _, trunk, picked, question = _schema(case, seed)

    def call(pairs, past=None, behind=()):
        keys = [p for _, p in behind] + [p for _, p in pairs]
        return _decoder(case, wt, [t for t, _ in pairs], [p for _, p in pairs], past, keys)

    def head(x):
        return x @ _f(wt["lm_head"]).T

    if case["kind"] == "prompt":
        pairs = sorted(trunk + [p for _, m in picked for p in m] + question, key=lambda p: p[1])
        pairs = [(t, i) for i, (t, _) in enumerate(pairs)]                  # positions are packed when nothing is cached
        return head(call(pairs)[0])[None]
    # every scaffold by itself: the trunk, and each picked member with the trunk around it
    kv, staged = call(trunk)[1], list(trunk)
    for at, own in picked:
        _, mine = call(trunk[:at] + own + trunk[at:])
        kv = [(torch.cat([k, a[at:at + len(own)]]), torch.cat([v, b[at:at + len(own)]])) for (k, v), (a, b) in zip(kv, mine)]
        staged += own
    x, new = call(question, kv, staged)
    if case["kind"] == "question":
        return head(x)[None]
    g = torch.Generator().manual_seed(seed * 53 + 3)
    out = []
    for t in torch.randint(4, VOCAB, (case["tokens"],), generator=g).tolist():
        kv = [(torch.cat([k, a]), torch.cat([v, b])) for (k, v), (a, b) in zip(kv, new)]
        staged += question
        question = [(t, question[-1][1] + 1)]
        x, new = call(question, kv, staged)
        out.append(head(x)[None])
    return out


def _exact_encode(case, seed):
    """The stores of all segments, in the order of ``run``: position, length, text."""
    wt = _decoder_weights(case, seed)
    out = []
    unions = case["unions"]
    trunk = _schema(case, seed)[2]

    def add(pairs, kv, a, b, key):
        out.append(((key[0], b - a, key[1]), torch.stack([torch.stack([k[a:b].transpose(0, 1), v[a:b].transpose(0, 1)]) for k, v in kv])))

    def call(pairs):
        return _decoder(case, wt, [t for t, _ in pairs], [p for _, p in pairs], None, [p for _, p in pairs])[1]

    def name(pairs):
        return Words().decode([t for t, _ in pairs]) if pairs[0][0] != 3 else " "

    root = call(trunk)
    at = 0
    for n in [case["text"]] + [case["doc_len"]] * case["docs"] + [1] * unions:
        add(trunk, root, at, at + n, (trunk[at][1], name(trunk[at:at + n])))
        at += n
    del root
    schema = _schema(case, seed)[0]
    for u in range(unions):
        before = case["text"] + case["docs"] * case["doc_len"] + u
        start = trunk[before - 1][1] + 1
        for m in range(case["members"]):
            body = re.search('<module name="u%d-%d">(.*?)</module>' % (u, m), schema).group(1)
            own = [(t, start + i) for i, t in enumerate(Words().encode(body))]
            kv = call(trunk[:before] + own)
            add(own, kv, before, before + len(own), (start, body))
    return [t for _, t in sorted(out, key=lambda o: o[0])]


def _turn_pairs(x, ang, mag=1.0):
    """Neighbouring columns turned by ``ang`` [n, pairs]; x [n, heads, 2 * pairs]."""
    c, s = (torch.cos(ang) * mag)[:, None], (torch.sin(ang) * mag)[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)


def _kazolorn(case, wt, tokens):
    w, h = case["width"], case["width"] // 128
    n, kv, eps = len(tokens), case["width"] // 512, 1e-6
    x = _f(wt["embed"][torch.tensor(tokens, device=DEV)])
    results = [x]
    pos = torch.arange(n, device=DEV, dtype=torch.float64)
    dist = pos[:, None] - pos[None]
    hidden = (dist < 0) | (dist >= 1024)
    slopes = torch.tensor([2.0 ** (-8.0 * (i + 1) / h) for i in range(h)], device=DEV, dtype=torch.float64)
    for i in range(4):
        p = {k[len("l%d." % i):]: _f(v) for k, v in wt.items() if k.startswith("l%d." % i)}
        z = _rms(x, eps) * p["norm1"]
        q = (z @ p["mix.q"].T + p["mix.q.b"]).view(n, h, 128)
        k = (z @ p["mix.k"].T + p["mix.k.b"]).view(n, kv, 128).repeat_interleave(h // kv, 1)
        s = torch.stack([q[:, j] @ k[:, j].T * 128 ** -0.5 - slopes[j] * dist for j in range(h)])
        s = (p["mix.talk"] @ s.reshape(h, -1)).view(h, n, n).masked_fill_(hidden, -math.inf)
        top = s.amax(-1, keepdim=True).clamp(min=0.0)
        e = torch.exp(s - top)
        e = e / (torch.exp(-top) + e.sum(-1, keepdim=True))
        a = torch.stack([e[j] @ k[:, j] for j in range(h)], 1).reshape(n, w)
        y = p["ls1"] * (a @ p["mix.o"].T + p["mix.o.b"])
        u = (_rms(x, eps) * p["norm2"]) @ p["mlp.up"].T
        c = p["mlp.act"]
        u = c[0] * _rms(u, eps) + c[1] * _rms(u * u, eps) + c[2] * _rms(u * u * u, eps) + c[3]
        y = y + p["ls2"] * (u @ p["mlp.down"].T)
        results.append(x + y)
        x = sum(c * r for c, r in zip(p["dwa"], results))
    return _rms(x, eps) * _f(wt["final.norm"])


def _fivesun(case, wt, tokens):
    w, h, kv, n, eps = case["width"], case["width"] // 128, case["width"] // 512, len(tokens), 1e-6
    x = _f(wt["embed"][torch.tensor(tokens, device=DEV)]) * w ** 0.5
    pos = torch.arange(n, device=DEV, dtype=torch.float64)
    dist = pos[:, None] - pos[None]
    block = torch.div(pos, 1024, rounding_mode="floor")
    first = None

    def attend(q, k, v, hidden, scale, sink=None):
        out = []
        for j in range(h):
            s = (q[:, j] @ k[:, j].T * scale).masked_fill_(hidden, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[j].expand(n, 1)], 1)
            out.append(torch.softmax(s, -1)[:, :n] @ v[:, j])
        return torch.stack(out, 1)

    def attention(z, p):
        nonlocal first
        ang = pos[:, None] * 1000000.0 ** (-torch.arange(0, 128, 2, device=DEV, dtype=torch.float64) / 128) / 4.0
        q = _turn_pairs(_rms((z @ p["q"].T).view(n, h, 128), eps) * p["q.norm"], ang)
        k = _turn_pairs(_rms((z @ p["k"].T).view(n, kv, 128), eps) * p["k.norm"], ang)
        v = _rms((z @ p["v"].T).view(n, kv, 128), eps)
        if first is None:
            first = v
        else:
            v = (1 - p["vmix"]) * v + p["vmix"] * first
        k, v = k.repeat_interleave(h // kv, 1), v.repeat_interleave(h // kv, 1)
        o = attend(q, k, v, (dist < 0) | (block[:, None] != block[None]), 128 ** -0.5, p["sink"])
        return (o * torch.sigmoid(z @ p["g"].T)[..., None]).reshape(n, w) @ p["o"].T

    def latent(z, p):
        rot, rank, base, factor, original = 64, 192, 10000.0, 8.0, 4096.0

        def pair(turns):
            return rot * math.log(original / (2 * math.pi * turns)) / (2 * math.log(base))
        lo, hi = max(math.floor(pair(32.0)), 0), min(math.ceil(pair(1.0)), rot - 1)
        f = base ** (-torch.arange(0, rot, 2, device=DEV, dtype=torch.float64) / rot)
        ramp = ((torch.arange(rot // 2, device=DEV, dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
        ang, mag = pos[:, None] * (f / factor * ramp + f * (1 - ramp)), 0.1 * math.log(factor) + 1
        q = (z @ p["q"].T).view(n, h, 128 + rot)
        down = z @ p["dkv"].T
        c = _rms(down[:, :rank], eps) * p["dkv.norm"]
        q = torch.cat([q[..., :128], _turn_pairs(q[..., 128:], ang, mag)], -1)
        kr = _turn_pairs(down[:, None, rank:], ang, mag).expand(n, h, rot)
        k = torch.cat([(c @ p["uk"].T).view(n, h, 128), kr], -1)
        o = attend(q, k, (c @ p["uv"].T).view(n, h, 128), (dist < 0) | (dist >= 1024), (128 + rot) ** -0.5)
        return (o.reshape(n, w) * torch.sigmoid(z @ p["g"].T)) @ p["o"].T

    def memory(z, p):
        q, k, v = ((z @ p[c].T).view(n, h, 128) for c in "qkv")
        q = q * 128 ** -0.5
        li = 10.0 * torch.tanh((z @ p["i"].T + p["i.b"]) / 10.0)
        lf = torch.nn.functional.logsigmoid(10.0 * torch.tanh((z @ p["f"].T + p["f.b"]) / 10.0))
        # the sum over earlier tokens written out: weight of token j at token t = exp(F_t - F_j + li_j - m_t), m from 0 at the start
        F = lf.cumsum(0).T
        a = F[:, :, None] - F[:, None] + li.T[:, None]
        a = a.masked_fill_(dist < 0, -math.inf)
        m = torch.maximum(a.amax(-1), F)
        e = torch.exp(a - m[..., None])
        s = torch.stack([q[:, j] @ k[:, j].T for j in range(h)]) * e
        den = torch.maximum(s.sum(-1).abs(), torch.exp(-m)) + 1e-6
        o = torch.stack([s[j] @ v[:, j] for j in range(h)]) / den[..., None]
        o = _rms(o.transpose(0, 1), eps).reshape(n, w) * p["norm"] * torch.sigmoid(z @ p["g"].T)
        return o @ p["o"].T

    def mlp(z, p):
        a = torch.relu(z @ p["gate"].T + p["gate.b"]) * (z @ p["up"].T + p["up.b"])
        return a @ p["down"].T + p["down.b"]

    for i, mixer in enumerate((attention, latent, attention, memory)):
        p = {k[len("l%d." % i):]: _f(v) for k, v in wt.items() if k.startswith("l%d." % i)}
        for which, f, part in (("1", mixer, "mix."), ("2", mlp, "mlp.")):
            z = _rms(x, eps) * p["norm" + which]
            y = f(z, {k[4:]: v for k, v in p.items() if k.startswith(part)}) * torch.sigmoid(z @ p["rg" + which].T + p["rg" + which + ".b"])
            x = x + _rms(y, eps) * p["norm" + which + "b"]
    return _rms(x, eps) * _f(wt["final.norm"])


def exact(case, seed):
    with torch.inference_mode():
        if case["kind"] == "encode":
            return _exact_encode(case, seed)
        if case["kind"] != "serve":
            return _exact_decoder(case, seed)
        wt = _served_weights(case, seed)
        model, p = _kazolorn if case["model"] == "kazolorn" else _fivesun, case["prompt"]
        head = _f(wt["head"])
        rows = [model(case, wt, toks)[p - 1:] @ head.T for toks in _requests(case, seed)]
        return [torch.stack([r[t] for r in rows]) for t in range(case["tokens"] + 1)]
