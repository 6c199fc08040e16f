"""Steps whose tables go up while earlier ones are still running: prompts and single tokens of several requests asked for without a wait between them give
what they give one at a time, and a step cannot be captured (its tables are new each time)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _model(name):
    if name == "kazolorn":
        from tests.test_gpu_kazolorn import model
        return model("mixed", torch.bfloat16)[2]
    from tests.test_gpu_fivesun import model
    return model("mixed", torch.bfloat16)[2]


@pytest.mark.parametrize("name", ["kazolorn", "fivesun"])
def test_steps_under_way_keep_their_own_tables(name):
    m, g = _model(name), torch.Generator().manual_seed(3)
    runs = [torch.randint(0, m.V, (int(n),), generator=g).tolist() for n in torch.randint(1, 60, (24,), generator=g)]

    arena = m.new_arena(1, 80)

    def one(tokens):
        slot = arena.alloc()
        out = [m.forward_rows(arena, [slot], [tokens])] + [m.forward_rows(arena, [slot], [[t]]) for t in tokens[:3]]
        arena.free(slot)
        return out

    one(runs[0])                                                   # (single tokens are a captured graph from here on)
    alone = []
    for r in runs:
        alone.append(one(r))
        torch.cuda.synchronize()
    busy = torch.randn(4096, 4096, device=DEV)
    for _ in range(40):                                            # (the stream is behind: all of the steps below wait for it)
        busy = busy @ busy * 1e-3
    under_way = [one(r) for r in runs]
    torch.cuda.synchronize()
    for a, b in zip(alone, under_way):
        assert all(torch.equal(x, y) for x, y in zip(a, b))


def test_a_step_is_not_captured():
    m = _model("kazolorn")
    arena = m.new_arena(1, 32)
    slot = arena.alloc()
    m.forward_rows(arena, [slot], [[1, 2, 3]])
    torch.cuda.synchronize()
    with pytest.raises(RuntimeError), torch.cuda.graph(torch.cuda.CUDAGraph()):
        m.forward_rows(arena, [slot], [[4, 5, 6]])
    torch.cuda.synchronize()
    assert m.forward_rows(arena, [slot], [[4, 5, 6]]).isfinite().all()
