"""An MPT call's inputs from the host (one upload of ids, positions and lengths) and from the device give the same logits, bit for bit: prompts, decoded
tokens, positions with gaps, several replays of one graph with other values, both ways in turn on the same graph."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_host_and_device_inputs_give_the_same_logits():
    from promptcache_amd.model.config import MptShape
    from promptcache_amd.model.mpt_hip import MptHIP
    from promptcache_amd.model.weights import make_mpt_weights_np
    shape = MptShape(vocab_size=512, hidden_size=256, num_hidden_layers=2, num_attention_heads=4)
    lm = MptHIP(shape, {k: torch.from_numpy(np.asarray(v)) for k, v in make_mpt_weights_np(shape, 3, 1.0).items()}, "cuda:0")
    g = torch.Generator().manual_seed(1)
    prompt = torch.randint(0, 512, (1, 40), generator=g)
    steps = [torch.randint(0, 512, (1, n), generator=g) for n in (3, 1, 1, 3, 1, 1)]

    def run(ways):
        pos = torch.arange(40)[None] * 2                         # every other position
        out = lm(input_ids=prompt, position_ids=pos, use_cache=True)
        logits = [out.logits]
        for t, way in zip(steps, ways):
            pos = torch.cat([pos, pos[:, -1:] + 3 + torch.arange(t.shape[1])[None]], 1)
            a, b = (t, pos) if way == "host" else (t.to("cuda:0"), pos.to("cuda:0")) if way == "device" else (t, pos.to("cuda:0"))
            out = lm(input_ids=a, position_ids=b, past_key_values=out.past_key_values, use_cache=True)
            logits.append(out.logits)
        return logits
    want = run(["device"] * 6)
    for ways in (["host"] * 6, ["host", "device"] * 3, ["host", "mixed"] * 3):
        for a, b in zip(run(ways), want):
            assert bool(torch.isfinite(a).all()) and torch.equal(a, b)


@pytest.mark.parametrize("rows", [65, 129, 288])
def test_qkv_in_slices_gives_what_one_launch_gives(rows, monkeypatch):
    """65 to 288 rows: q|k|v in two slices of K and the append behind them, against one launch."""
    from promptcache_amd.model.config import MptShape
    from promptcache_amd.model.mpt_hip import MptHIP
    from promptcache_amd.model.weights import make_mpt_weights_np
    shape = MptShape(vocab_size=512, hidden_size=512, num_hidden_layers=2, num_attention_heads=4)
    lm = MptHIP(shape, {k: torch.from_numpy(np.asarray(v)) for k, v in make_mpt_weights_np(shape, 3, 1.0).items()}, "cuda:0")
    assert lm.qkv_kslices(rows, lm.rows_kslices(rows, 512)) == 2
    ids = torch.randint(0, 512, (1, 40 + rows), generator=torch.Generator().manual_seed(rows))
    got = []
    for slices in ("2", "1"):
        monkeypatch.setenv("PC_ROWS_QKV_KS", slices)
        out = lm(input_ids=ids[:, :40], position_ids=torch.arange(40)[None], use_cache=True)
        got.append(lm(input_ids=ids[:, 40:], position_ids=torch.arange(40 + rows)[None], past_key_values=out.past_key_values, use_cache=True).logits.double())
        if hasattr(lm, "_graphs"):
            lm._graphs.clear()
    # (another order of fp32 sums moves one in a thousand keys, values and operands by their last fp16 bit: 2^-11 / sqrt(1000) of what they are part of)
    assert float((got[0] - got[1]).norm() / got[1].norm()) < 1e-4
