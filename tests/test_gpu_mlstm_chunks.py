"""pcb_mlstm_prompt and pcb_mlstm_step (the matrix memory in segments on the matrix cores, and one token per request; norm and gate included)
against the float64 recurrence: segments around the 16-row tiles and the 64-, 128- and 256-token forms, requests that resume, junk in the slots of
those that do not, forget gates that keep everything, that drop everything and that are closed for good."""
import pytest
import torch

from oracle import fivesun_oracle as O

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda:0", torch.float64


def rnd(*shape, seed=0, dtype=torch.float32):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV, dtype)


def rel(got, want):
    got, want = got.to("cpu", F64), want.to("cpu", F64)
    return float((got - want).norm() / want.norm())


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


# fp32 rows: the recurrence's own test holds token by token to 2e-5; products and sums here are fp32 as well.  bf16 rows: the inputs are exact either
# way, the results are rounded to 8 significant bits: 2^-8 of a value at most.
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("H,D,Dv,cap,seg,shift", [(2, 128, 128, 10.0, 64, 3.0), (2, 16, 24, 0.0, 64, 3.0), (4, 72, 128, 0.0, 128, -30.0),
                                                  (2, 128, 40, 4.0, 256, 6.0), (4, 8, 8, 0.0, 64, 0.0)])
def test_segments_and_steps_against_the_recurrence(H, D, Dv, cap, seg, shift, dtype, tol):
    from promptcache_amd import _blocks as B
    eps, rec = 1e-6, B.mlstm_state_floats(H, D, Dv)
    counts, starts, slots = [2 * seg + 2, 17, 1, seg, 16, seg - 1], [0, 9, 0, 4, 0, 7], [4, 0, 2, 6, 1, 5]
    n = sum(counts)
    N = 2 * H * D + 2 * H * Dv + 2 * H
    N = -(-N // 8) * 8
    P = rnd(n + 6, N, seed=1, dtype=dtype)                       # (the last six rows: one more token of every request)
    gf = P[:, 2 * H * D + H * Dv + H:2 * H * D + H * Dv + 2 * H]
    gf += shift
    if cap == 0.0:
        gf[5::11] = float("-inf")                                # nothing of what came before stays
    g0 = 2 * H * D + H * Dv + 2 * H
    gain, gate = 1 + 0.1 * rnd(H * Dv, seed=2), P[:, g0:g0 + H * Dv]
    state = rnd(7, rec, seed=3)
    state.view(7, H, -1)[..., -1] = 0.7
    f = lambda t: t.detach().to("cpu", F64)
    P6, s6 = f(P), f(state).view(7, H, -1)

    def oracle(rows, st):
        x, k = P6[rows], len(rows)
        q, kk, v = x[:, :H * D].view(k, H, D) * D ** -0.5, x[:, H * D:2 * H * D].view(k, H, D), x[:, 2 * H * D:2 * H * D + H * Dv].view(k, H, Dv)
        gi, gl = x[:, 2 * H * D + H * Dv:2 * H * D + H * Dv + H], x[:, 2 * H * D + H * Dv + H:g0]
        o, st = O.matrix_memory(q, kk, v, O.soft_cap(gi, cap), torch.nn.functional.logsigmoid(O.soft_cap(gl, cap)), st)
        return O.unit_rms(o, eps).reshape(k, H * Dv) * f(gain) * x[:, g0:g0 + H * Dv], st

    segs, chains, ends, row = [], [], [], 0
    for c, s0, slot in zip(counts, starts, slots):
        chains.append((slot, s0, len(segs), -(-c // seg)))
        for q in range(0, c, seg):
            segs.append((len(segs), 0, min(seg, c - q), row + q))
            ends.append(slot if q + seg >= c else -1)
        row += c
    ns = len(segs)
    cols = (P, P[:, H * D:], P[:, 2 * H * D:], P[:, 2 * H * D + H * Dv:], P[:, 2 * H * D + H * Dv + H:])
    out = torch.zeros(n + 6, H * Dv, device=DEV, dtype=dtype)
    nan = lambda *s: torch.full(s, float("nan"), device=DEV)
    tail = (H, D, Dv, D ** -0.5, cap, gain, gate, N, out, eps)
    assert B.mlstm_prompt_fits(D, Dv, N, cols, gate, seg) and B.mlstm_step_fits(D, Dv, N, cols[2])
    untouched = state[3].clone()
    B.mlstm_prompt(cols, N, i32(segs), ns, i32(chains), len(chains), seg, i32(ends), state, *tail, nan(ns, rec), nan(ns, H), nan(ns, rec))
    want, after, row = [], [], 0
    for c, s0, slot in zip(counts, starts, slots):
        st = (s6[slot][:, :D * Dv].reshape(H, D, Dv), s6[slot][:, D * Dv:D * Dv + D], s6[slot][:, -1]) if s0 else None
        o, st = oracle(list(range(row, row + c)), st)
        want.append(o), after.append(st)
        got = state[slot].view(H, -1)
        assert rel(got[:, :D * Dv].reshape(H, D, Dv), st[0]) < 2e-5 and rel(got[:, D * Dv:-1], st[1]) < 2e-5
        assert torch.allclose(f(got[:, -1]), st[2], rtol=1e-5, atol=1e-5)
        row += c
    assert rel(out[:n], torch.cat(want)) < tol and torch.equal(state[3], untouched)
    # one more token each
    B.mlstm_step(cols, N, i32([(s, s0 + c, 1, n + b) for b, (s, s0, c) in enumerate(zip(slots, starts, counts))]), 6, state, *tail)
    for b, slot in enumerate(slots):
        o, st = oracle([n + b], after[b])
        got = state[slot].view(H, -1)
        assert rel(out[n + b], o[0]) < tol and rel(got[:, :D * Dv].reshape(H, D, Dv), st[0]) < 2e-5 and rel(got[:, D * Dv:-1], st[1]) < 2e-5
    # a first token: the slot's junk is not read
    B.mlstm_step(cols, N, i32([(3, 0, 1, n)]), 1, state, *tail)
    assert rel(out[n], oracle([n], None)[0][0]) < tol


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,Dv", [(200, 100), (60, 252)])
def test_steps_of_wide_heads(D, Dv, dtype):
    from promptcache_amd import _blocks as B
    H, eps = 3, 1e-6
    N = 2 * H * D + H * Dv + 2 * H + 2
    P, state = rnd(5, N, seed=1, dtype=dtype), rnd(5, B.mlstm_state_floats(H, D, Dv), seed=2)
    state.view(5, H, -1)[..., -1] = 0.2
    cols = (P, P[:, H * D:], P[:, 2 * H * D:], P[:, 2 * H * D + H * Dv:], P[:, 2 * H * D + H * Dv + H:])
    reqs, ref = i32([(4, 3, 1, 0), (1, 0, 1, 1), (0, 8, 1, 4)]), state.clone()
    out, raw, want = (torch.zeros(5, H * Dv, device=DEV, dtype=t) for t in (dtype, torch.float32, dtype))
    B.mlstm(*cols, N, reqs, 3, ref, H, D, Dv, D ** -0.5, 5.0, raw)
    B.gated_norm(raw, None, None, 0, want, eps, 5, group=Dv)
    assert B.mlstm_step_fits(D, Dv, N, cols[2])
    B.mlstm_step(cols, N, reqs, 3, state, H, D, Dv, D ** -0.5, 5.0, None, None, 0, out, eps)
    assert rel(state, ref) < 1e-6 and rel(out, want) < (1e-5 if dtype == torch.float32 else 2.0 ** -8)


def layer(H, D, Dv, n, dtype, shift=3.0):
    """Columns of n random tokens, their strides' row length, gate and gain."""
    N = -(-(2 * H * D + 2 * H * Dv + 2 * H) // 8) * 8
    P = rnd(n, N, seed=1, dtype=dtype)
    P[:, 2 * H * D + H * Dv + H:2 * H * D + H * Dv + 2 * H] += shift
    g0 = 2 * H * D + H * Dv + 2 * H
    return (P, P[:, H * D:], P[:, 2 * H * D:], P[:, 2 * H * D + H * Dv:], P[:, 2 * H * D + H * Dv + H:]), N, P[:, g0:g0 + H * Dv], 1 + 0.1 * rnd(H * Dv, seed=2)


def one_prompt(cols, N, H, D, Dv, n, seg, state, slot, pos0, gain, gate):
    from promptcache_amd import _blocks as B
    rec, starts = B.mlstm_state_floats(H, D, Dv), range(0, n, seg)
    ns, nan = len(starts), lambda *s: torch.full(s, float("nan"), device=DEV)
    out = torch.zeros(n, H * Dv, device=DEV, dtype=cols[0].dtype)
    B.mlstm_prompt(cols, N, i32([(i, 0, min(seg, n - q), q) for i, q in enumerate(starts)]), ns, i32([(slot, pos0, 0, ns)]), 1, seg,
                   i32([-1] * (ns - 1) + [slot]), state, H, D, Dv, D ** -0.5, 0.0, gain, gate, N, out, 1e-6, nan(ns, rec), nan(ns, H), nan(ns, rec))
    return out


# (bounds as above)
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2.0 ** -8)])
@pytest.mark.parametrize("closed", ["one token", "the first token", "a whole segment", "a last segment of one token", "every token", "every other token"])
@pytest.mark.parametrize("pos0", [0, 5])
def test_closed_input_gates(closed, pos0, dtype, tol):
    from promptcache_amd import _blocks as B
    H, D, Dv, seg = 2, 64, 40, 32
    n = 2 * seg + 1
    cols, N, gate, gain = layer(H, D, Dv, n, dtype)
    shut = {"one token": [5], "the first token": [0], "a whole segment": range(seg, 2 * seg), "a last segment of one token": [2 * seg], "every token": range(n),
            "every other token": range(1, n, 2)}[closed]
    cols[3][list(shut), :H] = float("-inf")
    state = rnd(2, B.mlstm_state_floats(H, D, Dv), seed=3)
    state.view(2, H, -1)[..., -1] = 0.7
    f = lambda t: t.detach().to("cpu", F64)
    s6, x = f(state[1]).view(H, -1), [f(c) for c in cols]
    st = (s6[:, :D * Dv].reshape(H, D, Dv), s6[:, D * Dv:-1], s6[:, -1]) if pos0 else None
    o, (S, nv, m) = O.matrix_memory(x[0][:, :H * D].view(n, H, D) * D ** -0.5, x[1][:, :H * D].view(n, H, D), x[2][:, :H * Dv].view(n, H, Dv), x[3][:, :H],
                                    torch.nn.functional.logsigmoid(x[4][:, :H]), st)
    want = O.unit_rms(o, 1e-6).reshape(n, H * Dv) * f(gain) * f(gate)
    got = f(one_prompt(cols, N, H, D, Dv, n, seg, state, 1, pos0, gain, gate))
    near = lambda a, b, t: bool(torch.isfinite(a).all()) and float((a - b).norm()) <= t * float(b.norm())      # (from nothing, no token: all zeros)
    after = f(state[1]).view(H, -1)
    assert near(got, want, tol)
    assert near(after[:, :D * Dv].reshape(H, D, Dv), S, 2e-5) and near(after[:, D * Dv:-1], nv, 2e-5) and torch.allclose(after[:, -1], m, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("at", [0, 7, 15, 16, 37, 49])
def test_a_value_that_is_no_number_leaves_earlier_rows_alone(at, bad, dtype):
    from promptcache_amd import _blocks as B
    H, D, Dv, n = 2, 64, 72, 50
    cols, N, gate, gain = layer(H, D, Dv, n, dtype)
    rec = B.mlstm_state_floats(H, D, Dv)
    clean = one_prompt(cols, N, H, D, Dv, n, 64, torch.zeros(2, rec, device=DEV), 1, 0, gain, gate)
    cols[2][at, Dv + 3] = bad                                    # (head 1)
    got = one_prompt(cols, N, H, D, Dv, n, 64, torch.zeros(2, rec, device=DEV), 1, 0, gain, gate)
    # the rows in front of it and the other head: to the rounding of sums in another order
    assert bool(torch.isfinite(got[:at]).all()) and bool(torch.isfinite(got[:, :Dv]).all()) and not bool(torch.isfinite(got[at:, Dv + 3]).any())
    assert rel(got[:, :Dv], clean[:, :Dv]) == 0 and (at == 0 or rel(got[:at], clean[:at]) < (1e-6 if dtype == torch.float32 else 2.0 ** -9))


@pytest.mark.parametrize("shut", [[0], [40], [32, 33, 50], range(32, 64), range(65)])
@pytest.mark.parametrize("pos0", [0, 5])
def test_closed_input_gates_token_by_token(shut, pos0):
    """The segments of sizes that the matrix cores' kernels do not take: from nothing, chained, each from its start."""
    from promptcache_amd import _blocks as B
    H, D, Dv, seg, n = 2, 136, 40, 32, 65
    cols, N, _, _ = layer(H, D, Dv, n, torch.float32)
    cols[3][list(shut), :H] = float("-inf")
    rec, f = B.mlstm_state_floats(H, D, Dv), lambda t: t.detach().to("cpu", F64)
    state = rnd(2, rec, seed=3)
    state.view(2, H, -1)[..., -1] = 0.7
    s6, x = f(state[1]).view(H, -1), [f(c) for c in cols]
    st = (s6[:, :D * Dv].reshape(H, D, Dv), s6[:, D * Dv:-1], s6[:, -1]) if pos0 else None
    want, (S, nv, m) = O.matrix_memory(x[0][:, :H * D].view(n, H, D) * D ** -0.5, x[1][:, :H * D].view(n, H, D), x[2][:, :H * Dv].view(n, H, Dv), x[3][:, :H],
                                       torch.nn.functional.logsigmoid(x[4][:, :H]), st)
    local, start, fsum, out = torch.empty(3, rec, device=DEV), torch.empty(3, rec, device=DEV), torch.empty(3, H, device=DEV), torch.zeros(n, H * Dv, device=DEV)
    tail = (H, D, Dv, D ** -0.5, 0.0)
    B.mlstm(*cols, N, i32([(g, 0, min(seg, n - g * seg), g * seg) for g in range(3)]), 3, local, *tail, None, from_nothing=True, log_f_sum=fsum)
    B.mlstm_chain(local, fsum, start, state, i32([(1, pos0, 0, 3)]), 1, H, D, Dv)
    B.mlstm(*cols, N, i32([(g, 1, min(seg, n - g * seg), g * seg) for g in range(3)]), 3, start, *tail, out, end_slots=i32([-1, -1, 1]), end_state=state)
    near = lambda a, b: bool(torch.isfinite(a).all()) and float((a - b).norm()) <= 2e-5 * float(b.norm())
    after = f(state[1]).view(H, -1)
    assert near(f(out), want.reshape(n, H * Dv)) and near(after[:, :D * Dv].reshape(H, D, Dv), S) and near(after[:, D * Dv:-1], nv)
    assert torch.allclose(after[:, -1], m, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-5), (torch.bfloat16, 2e-5)])
@pytest.mark.parametrize("H,D,Dv,R,count", [(8, 16, 128, 200, 3), (16, 40, 70, 80, 9), (4, 136, 200, 96, 2), (3, 8, 300, 24, 1)])
def test_more_workgroups_than_run_at_once(H, D, Dv, R, count, dtype, tol):
    """Several blocks of value columns share a head's n and m, which move in place: a block that starts when another one has ended must not see them moved.
    (Against each request by itself: launches that the chip has room for.)"""
    from promptcache_amd import _blocks as B
    n = R * count
    cols, N, _, _ = layer(H, D, Dv, n, dtype)
    rec = B.mlstm_state_floats(H, D, Dv)
    state = rnd(R, rec, seed=3)
    state.view(R, H, -1)[..., -1] = 0.7
    ref, out, want = state.clone(), torch.zeros(n, H * Dv, device=DEV), torch.zeros(n, H * Dv, device=DEV)
    tail = (H, D, Dv, D ** -0.5, 0.0)
    reqs = [(r, 5, count, r * count) for r in range(R)]
    B.mlstm(*cols, N, i32(reqs), R, state, *tail, out)
    for r in reqs:
        B.mlstm(*cols, N, i32([r]), 1, ref, *tail, want)
    assert torch.equal(out, want) and torch.equal(state, ref)
    # ... and a few of them against the recurrence
    f = lambda t: t.detach().to("cpu", F64)
    s0, x = rnd(R, rec, seed=3), [f(c) for c in cols]
    s0.view(R, H, -1)[..., -1] = 0.7
    for r in (0, R // 2, R - 1):
        rows, s6 = slice(r * count, (r + 1) * count), f(s0[r]).view(H, -1)
        o, (S, nv, m) = O.matrix_memory(x[0][rows, :H * D].view(count, H, D) * D ** -0.5, x[1][rows, :H * D].view(count, H, D),
                                        x[2][rows, :H * Dv].view(count, H, Dv), x[3][rows, :H], torch.nn.functional.logsigmoid(x[4][rows, :H]),
                                        (s6[:, :D * Dv].reshape(H, D, Dv), s6[:, D * Dv:-1], s6[:, -1]))
        after = f(state[r]).view(H, -1)
        assert rel(f(out[rows]), o.reshape(count, H * Dv)) < tol and rel(after[:, :D * Dv].reshape(H, D, Dv), S) < tol and rel(after[:, D * Dv:-1], nv) < tol
