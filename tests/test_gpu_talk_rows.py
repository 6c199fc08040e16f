"""pcb_attn_talk_rows (single rows of the attention with talking heads, one launch) against float64: rows whose keys end around the 64-key blocks and
around what one workgroup takes, windows, no window, every number of heads to a key head, and what the general form does with NaN."""
import pytest
import torch

from oracle import kazolorn_oracle as O

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


def B():
    from promptcache_amd import _blocks
    return _blocks


def rel(got, want):
    got, want = got.to("cpu", F64), want.to("cpu", F64)
    return float((got - want).norm() / want.norm())


def case(dtype, H, G, D, window, places, seed=0):
    """One row per place (its position) in slots 2, 1, 0, 2 + 1, ..: queries, cache, tiles; flat rows in reverse order."""
    g = torch.Generator().manual_seed(seed)
    n, cap = len(places), max(places) + 4
    q = torch.randn(n, H * D, generator=g).to(dtype)
    cache = torch.randn(n, G, cap, D, generator=g).to(dtype)
    talk = torch.eye(H) + 0.2 * torch.randn(H, H, generator=g)
    tiles = torch.tensor([[n - 1 - b, p, 1, n - 1 - b] for b, p in enumerate(places)], dtype=torch.int32)
    want = torch.stack([O.talking_attention(q[n - 1 - b].view(1, H, D).to(F64), cache[n - 1 - b, :, :p + 1].transpose(0, 1).to(F64), 0.3, window,
                                            talk.to(F64), first_pos=p).reshape(H * D) for b, p in enumerate(places)]).flip(0)
    return q.to(DEV), cache.to(DEV), talk.to(DEV), tiles.to(DEV), cap, want


def attend(q, cache, talk, tiles, cap, H, G, D, window, slopes, sink, counters):
    n = tiles.shape[0]
    out = torch.zeros_like(q)
    part = torch.full((B().attn_talk_rows_part(n, H, D),), float("nan"), device=DEV)
    B().attn_talk_rows(q, tiles.reshape(-1), n, cache, G * cap * D, cap * D, H, G, D, 0.3, window, cap, slopes, talk, sink, part, counters, out)
    return out


# the bounds of the general form's tests; fp32 sums run over up to 2 100 keys here
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 4e-6), (torch.bfloat16, 1.5e-2)])
@pytest.mark.parametrize("H,G,D,window,places", [
    (16, 4, 128, 1024, [0, 1, 62, 63, 64, 127, 128, 1022, 1023, 1024, 1500]),
    (8, 2, 128, 0, [5, 2100, 1030, 63]),          # no window: workgroups of 192 keys
    (4, 1, 128, 100, [37, 99, 100, 250]),
    (32, 4, 64, 70, [200, 69, 3]),                # eight heads to a key head, the most heads
    (12, 6, 40, 33, [20, 200, 31, 32, 33]),       # two to one, columns in chunks of eight only
    (3, 3, 8, 1, [0, 9]),                         # a window of one key
    (24, 24, 72, 65, [64, 65, 300]),
])
def test_single_rows_against_the_oracle(H, G, D, window, places, dtype, tol):
    assert B().attn_talk_rows_fits(dtype, H, G, D)
    q, cache, talk, tiles, cap, want = case(dtype, H, G, D, window, places)
    slopes = O.head_slopes(H).float().to(DEV)
    counters = torch.zeros(len(places), dtype=torch.int32, device=DEV)
    got = attend(q, cache, talk, tiles, cap, H, G, D, window, slopes, True, counters)
    assert rel(got, want) < tol
    for r in range(len(places)):
        assert rel(got[r], want[r]) < 2 * tol, places[::-1][r]
    # counters are left as they were found; a merged row does not depend on who came last
    for _ in range(5):
        assert torch.equal(attend(q, cache, talk, tiles, cap, H, G, D, window, slopes, True, counters), got)
    assert not bool(counters.any())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("sink,mixed", [(True, False), (False, True), (False, False)])
def test_single_rows_as_the_general_form_gives_them(dtype, sink, mixed):
    H, G, D, window, places = 8, 2, 32, 0, [1200, 40, 64, 1]
    q, cache, talk, tiles, cap, _ = case(dtype, H, G, D, window, places)
    talk = talk if mixed else None
    counters = torch.zeros(4, dtype=torch.int32, device=DEV)
    scratch = torch.empty(4 * 16 * H * B().attn_talk_band(window, cap), device=DEV)

    def general(x):
        out = torch.zeros_like(x)
        B().attn_talk(x, tiles.reshape(-1), 4, cache, G * cap * D, cap * D, H, G, D, 0.3, window, cap, None, talk, sink, scratch, out, max_tile_rows=1)
        return out
    got = attend(q, cache, talk, tiles, cap, H, G, D, window, None, sink, counters)
    assert rel(got, general(q)) < (2e-6 if dtype == torch.float32 else 2.0 ** -8)      # (bf16: both round the same numbers once)
    # rows that are no numbers stay none, the others keep their bits
    x = q.clone()
    x[0, 3], x[2, 40] = float("nan"), float("inf")
    bad = attend(x, cache, talk, tiles, cap, H, G, D, window, None, sink, counters)
    assert torch.equal(torch.isnan(bad), torch.isnan(general(x))) and torch.equal(bad[[1, 3]], got[[1, 3]]) and bool(torch.isnan(bad[[0, 2]]).any())


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 4e-6), (torch.bfloat16, 1.5e-2)])
@pytest.mark.parametrize("n,places", [(1, [3300]), (4, [3071, 3072, 64, 7000]), (5, [3300, 0, 1023, 1024, 4100]), (49, [1024 + 61 * b for b in range(49)])])
def test_a_rows_share_of_workgroups_does_not_depend_on_the_capacity(n, places, dtype, tol):
    """Eight, sixteen and 32 workgroups to a row; launched for a cache much longer than any row, as captured steps are, and for the longest row."""
    H, G, D = 4, 2, 64
    q, cache, talk, tiles, cap, want = case(dtype, H, G, D, 0, places)
    slopes, out = O.head_slopes(H).float().to(DEV), []
    counters = torch.zeros(n, dtype=torch.int32, device=DEV)
    for longest in (max(places) + 1, 1 << 20):
        got, part = torch.zeros_like(q), torch.full((B().attn_talk_rows_part(n, H, D),), float("nan"), device=DEV)
        B().attn_talk_rows(q, tiles.reshape(-1), n, cache, G * cap * D, cap * D, H, G, D, 0.3, 0, longest, slopes, talk, True, part, counters, got)
        assert rel(got, want) < tol and not bool(counters.any())
        out.append(got)
        used = part.view(n, -1, H * D + 2 * H).isfinite().all(-1).sum(1)
        for r, p in enumerate(places):                           # (records that a row's workgroups left: none from one alone)
            blocks = p // 64 + 1
            most = 8 if n > 48 else 32 if n <= 4 and blocks > 48 else 16
            per = -(-blocks // most)
            assert int(used[r]) == (0 if blocks <= per else -(-blocks // per)), (r, p)
    assert torch.equal(out[0], out[1])
