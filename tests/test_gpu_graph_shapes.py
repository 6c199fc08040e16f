"""Captured forwards over one arena behind prompts of different staged lengths: each replays a graph whose attention launches have the shape that its own length asks
for, so what ran before neither changes a result's bits nor makes a long cache be walked by the few streams of a short one."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DOCS = (630, 670)          # staged: ~640 rows (three streams of keys at 32 heads) and ~1310 (all seven); the workspaces of both are the same size


def _engine(kind):
    from promptcache_amd import CacheEngine
    from promptcache_amd.model import Llama2, Mpt
    from promptcache_amd.model.config import LlamaShape, MptShape
    from promptcache_amd.model.weights import make_mpt_weights_np, make_weights_np
    if kind == "llama":
        shape = LlamaShape(vocab_size=512, hidden_size=4096, intermediate_size=256, num_hidden_layers=1, num_attention_heads=32, num_key_value_heads=32)
        lm = Llama2(name="t", shape=shape, weights=make_weights_np(shape, 1, 0.3), device="cuda:0")
    else:
        shape = MptShape(vocab_size=512, hidden_size=4096, num_hidden_layers=1, num_attention_heads=32)
        lm = Mpt(name="t", shape=shape, weights=make_mpt_weights_np(shape, 1, 0.3), device="cuda:0")
    return lm, CacheEngine(3072, lm)


def _ask(lm, eng, docs, rows):
    """A question over the first ``docs`` modules, a schema of its own for each number (modules are staged in the order of their use)."""
    from promptcache_amd import Prompt, synth
    name = "gs%d" % docs
    if name not in eng.schemas:
        mods = "".join('<module name="m%d">%s</module>' % (i, synth.words(n, 2 + i)) for i, n in enumerate(DOCS[:docs]))
        eng.add_schema('<schema name="%s">%s%s</schema>' % (name, synth.words(12, 1), mods))
    eng.prompt_cache.reset()
    prompt = Prompt('<prompt schema="%s">%s%s</prompt>' % (name, "".join("<m%d/>" % i for i in range(docs)), synth.words(rows - 1, 9)))
    ids, pos, _, cache = eng.process(prompt, return_full_position_ids=lm.use_full_position_ids)
    out = lm(input_ids=torch.tensor([ids]), position_ids=torch.tensor([pos]), past_key_values=cache, use_cache=True)
    return out.logits.clone(), len(ids), len(eng.prompt_cache)


@pytest.mark.parametrize("kind", ["llama", "mpt"])
@pytest.mark.parametrize("rows", [14, 27])
def test_a_graph_is_replayed_at_its_own_launch_shape_only(kind, rows):
    alone = {}
    for docs in (1, 2):
        lm, eng = _engine(kind)
        alone[docs], asked, staged = _ask(lm, eng, docs, rows)
        assert (asked > 16) == (rows == 27) and 3 <= asked <= 32 and (600 < staged <= 690 if docs == 1 else 1275 <= staged < 1380)
    for first in (1, 2):
        lm, eng = _engine(kind)
        for docs in (first, 3 - first, first):
            got, _, _ = _ask(lm, eng, docs, rows)
            assert torch.equal(got, alone[docs])
