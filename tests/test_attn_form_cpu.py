"""What stands for an attention launch in a captured forward's key (pc_attn_form), without a GPU: lengths whose launches differ have different ones, lengths whose launches
are alike the same one."""
import pytest


def _n():
    from promptcache_amd import _native
    return _native


# (heads, rows, staged lengths of one launch, lengths of others)
@pytest.mark.parametrize("H,rows,alike,others", [
    (32, 16, (300, 650, 768), (769, 1024, 1025, 1300, 8000)),        # three streams / five / seven
    (32, 16, (769, 1024), (768, 1025)),
    (32, 16, (1025, 1265, 2096, 8000), (100, 650)),
    (32, 4, (300, 768), (769, 1024)),
    (32, 4, (769, 1024, 5000), (300,)),
    (32, 2, (300, 769, 5000), (250,)),                               # (250 and two rows: not the kernel of few rows)
    (32, 27, (300, 768), (769, 1300)),                               # a row tile a workgroup / two in one
    (40, 16, (650, 700), (1300, 8199)),
    (40, 27, (300, 768), (769, 3000)),
])
@pytest.mark.parametrize("alibi", [0, 1])
def test_lengths_of_one_launch(H, rows, alike, others, alibi):
    n = _n()
    mine = {n.attn_form(1, H, 128, rows, p, -1, alibi) for p in alike}
    assert len(mine) == 1 and 0 not in mine
    for p in others:
        assert n.attn_form(1, H, 128, rows, p, -1, alibi) not in mine


def test_the_size_of_the_workspace_does_not_tell():
    n = _n()
    assert n.attn_workspace_bytes(1, 32, 128, 16, 650 + 16) == n.attn_workspace_bytes(1, 32, 128, 16, 1300 + 16)
    assert n.attn_form(1, 32, 128, 16, 650, -1) != n.attn_form(1, 32, 128, 16, 1300, -1)


def test_every_launch_fits_its_workspace_and_modes_differ():
    n = _n()
    for H in (4, 8, 32, 40, 71):
        for rows in (1, 2, 5, 16, 17, 32, 33, 64, 128, 259, 512):
            for past in (0, 1, 63, 255, 256, 768, 769, 1024, 1025, 2047, 6143, 6144, 9000):
                for lo in (0, -1, -2):
                    for alibi in (0, 1):
                        splits = n.attn_form(1, H, 128, rows, past, lo, alibi) & 255
                        assert splits >= 1
                        if splits > 1:
                            assert n.attn_workspace_bytes(1, H, 128, rows, past + rows) >= H * splits * rows * 130 * 4
    assert n.attn_form(1, 32, 128, 12, 1700, -1) != n.attn_form(1, 32, 128, 12, 1700, 0)
    for bad in ((0, 32, 128, 1, 1), (1, 0, 128, 1, 1), (1, 32, 96, 1, 1), (1, 32, 128, 0, 1), (1, 32, 128, 1, -1)):
        assert n.attn_form(*bad, 0) == 0


@pytest.mark.parametrize("H,past", [(28, 2048), (32, 1792), (40, 1280), (64, 768)])
def test_positions_in_a_chain_of_tiles(H, past):
    """17 to 32 rows with ALiBi leave the kernel of few rows where a wave has a second tile (head dim 128)."""
    n = _n()
    plain = n.attn_form(1, H, 128, 27, past, -1, 0), n.attn_form(1, H, 128, 27, past + 1, -1, 0)
    alibi = n.attn_form(1, H, 128, 27, past, -1, 1), n.attn_form(1, H, 128, 27, past + 1, -1, 1)
    assert alibi[0] == plain[0] and plain[1] == plain[0] and alibi[1] != alibi[0]
    assert n.attn_form(1, H, 64, 27, past + 1, -1, 1) == n.attn_form(1, H, 64, 27, past, -1, 1)
    assert n.attn_form(1, H, 128, 16, past + 1, -1, 1) == n.attn_form(1, H, 128, 16, past, -1, 1)
