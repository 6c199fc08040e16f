"""An MPT question whose staging is left to the forward: the same logits as with the copy inside ``process``, bit for bit; the rows are there for whoever looks
first; a staging that another one replaces is never carried out."""
import pytest
import torch

pytestmark = pytest.mark.gpu
MODULES = "".join('<module name="d%d">%s</module>' % (d, " ".join("w%d" % ((7 * i + 31 * d) % 400) for i in range(n))) for d, n in enumerate((5, 70, 33)))
SCHEMA = '<schema name="s">w1 w2 w3 %s</schema>' % MODULES


class Words:
    unk_token, unk_token_id, bos_token_id, eos_token, eos_token_id = "<unk>", 0, 1, "</s>", 2

    def encode(self, text, add_special_tokens=False):
        return [4 + int(w[1:]) for w in text.split()]

    def decode(self, ids, **_):
        return " ".join("w%d" % (i - 4) for i in ids)


@pytest.mark.parametrize("question", ["w9", " ".join("w%d" % i for i in range(40)), " ".join("w%d" % (i % 300) for i in range(90))])
def test_left_to_the_forward(question):
    from promptcache_amd import CacheEngine, Prompt
    from promptcache_amd.model import Mpt
    from promptcache_amd.model.config import MptShape
    from promptcache_amd.model.weights import make_mpt_weights_np
    shape = MptShape(vocab_size=512, hidden_size=512, num_hidden_layers=2, num_attention_heads=4)
    lm = Mpt(shape=shape, weights={k: torch.from_numpy(v) for k, v in make_mpt_weights_np(shape, 3, 1.0).items()}, tokenizer=Words(), device="cuda:0")
    engine = CacheEngine(512, lm)
    engine.add_schema(SCHEMA)
    cache = engine.prompt_cache
    assert cache.defer_gather
    prompts = [Prompt('<prompt schema="s">%s%s</prompt>' % (refs, question)) for refs in ("<d0/><d1/><d2/>", "<d1/>", "<d2/><d0/>")]

    def ask(prompt, defer, look=False):
        cache.defer_gather = defer
        cache.reset()
        cache.arena.buf.fill_(float("nan"))                          # (what a forward reads has been staged for it)
        for s in engine.schemas["s"].cache_l1.values():
            s.usage_counter = 0
        ids, pos, _, past = engine.process(prompt, return_full_position_ids=True)
        assert (cache.arena.pending is not None) == defer
        if look:
            k, v = past[0]
            assert bool(torch.isfinite(k[..., :len(cache), :]).all()) and cache.arena.pending is None
        out = lm(input_ids=torch.tensor([ids]), position_ids=torch.tensor([pos]), past_key_values=past, use_cache=True)
        assert cache.arena.pending is None
        return out.logits
    for p in prompts + prompts[:1]:
        want = ask(p, False)
        assert bool(torch.isfinite(want).all())
        assert torch.equal(ask(p, True), want) and torch.equal(ask(p, True, look=True), want)
    # the second of two stagings counts
    cache.defer_gather = True
    cache.reset()
    engine.process(prompts[0], return_full_position_ids=True)
    assert torch.equal(ask(prompts[1], True), ask(prompts[1], False))
