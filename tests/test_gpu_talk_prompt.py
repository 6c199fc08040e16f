"""pcb_attn_talk's single pass for bf16 prompts (four query heads of 128 columns to a key head) against float64: rows around its units of 4, 8 and 16
queries, keys around its tiles of 64, windows, prompts behind cached keys, tiles of 16 and of 64 rows, and numbers that are none."""
import pytest
import torch

from oracle import kazolorn_oracle as O

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


def attend(q, cache, lens, first, talk, slopes, sink, window, wide):
    """Requests b of lens[b] rows from position first[b] on, in slot b; ``wide``: with the second tile table."""
    from promptcache_amd import _blocks as B
    (m, H, D), (_, G, cap, _) = q.shape, cache.shape

    def table(step):
        out, row = [], 0
        for b, (n, f) in enumerate(zip(lens, first)):
            out += [[b, f + at, min(step, n - at), row + at] for at in range(0, n, step)]
            row += n
        return torch.tensor(out, dtype=torch.int32, device=DEV)
    t16, t64 = table(16), table(64)
    scratch = torch.empty(t16.shape[0] * 16 * H * B.attn_talk_band(window, cap), device=DEV)
    out = torch.full((m + 1, H * D), 7.0, device=DEV, dtype=q.dtype)
    B.attn_talk(q.reshape(m, H * D), t16.reshape(-1), t16.shape[0], cache, G * cap * D, cap * D, H, G, D, 0.3, window, cap, slopes, talk, sink, scratch, out,
                tiles64=t64.reshape(-1) if wide else None, n_tiles64=t64.shape[0])
    assert bool((out[m] == 7.0).all())                           # rows past the last are not touched
    return out[:m].view(m, H, D)


@pytest.mark.parametrize("H", [4, 8, 16])
@pytest.mark.parametrize("window,lens,first", [
    (1024, [5, 8, 9, 31, 33], [0, 0, 70, 1, 1100]),
    (0, [64, 65, 63], [0, 200, 1]),
    (70, [150, 17], [0, 500]),
    (1, [20], [3]),
])
def test_prompts_against_the_oracle(H, window, lens, first):
    g = torch.Generator().manual_seed(H)
    m, G, cap = sum(lens), H // 4, max(n + f for n, f in zip(lens, first)) + 3
    q, cache = torch.randn(m, H, 128, generator=g).bfloat16(), torch.randn(len(lens), G, cap, 128, generator=g).bfloat16()
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    slopes = O.head_slopes(H).float()
    at, want = 0, []
    for b, (n, f) in enumerate(zip(lens, first)):
        want.append(O.talking_attention(q[at:at + n].to(F64), cache[b, :, :f + n].transpose(0, 1).to(F64), 0.3, window, talk.to(F64), first_pos=f))
        at += n
    want = torch.cat(want).reshape(m, H, 128)
    for wide in (True, False):
        got = attend(q.to(DEV), cache.to(DEV), lens, first, talk.to(DEV), slopes.to(DEV), True, window, wide).to("cpu", F64)
        # results are rounded to 8 bits once (2^-9 of each, 1.1e-3 in the norm); weights carry 16
        assert float((got - want).norm() / want.norm()) < 2e-3
        worst = ((got - want).norm(dim=(1, 2)) / want.norm(dim=(1, 2))).max()
        assert float(worst) < 4e-3


@pytest.mark.parametrize("H", [4, 8, 16])
def test_rows_that_are_no_numbers_stay_alone(H):
    g = torch.Generator().manual_seed(1)
    n, G = 50, H // 4
    q, cache = torch.randn(n, H, 128, generator=g).bfloat16().to(DEV), torch.randn(1, G, 60, 128, generator=g).bfloat16().to(DEV)
    talk = (torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)).to(DEV)
    for sink in (True, False):
        clean = attend(q, cache, [n], [0], talk, None, sink, 0, True)
        x = q.clone()
        x[3, 1, 5], x[30, H - 1, 100] = float("nan"), float("inf")
        bad = attend(x, cache, [n], [0], talk, None, sink, 0, True)
        keep = [r for r in range(n) if r not in (3, 30)]
        assert torch.equal(bad[keep], clean[keep]) and bool(torch.isnan(bad[3]).all()) and bool(torch.isnan(bad[30]).any())
