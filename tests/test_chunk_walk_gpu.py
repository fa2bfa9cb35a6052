"""The walk of a recurrence by chunks of 16 rows (csrc/recurrence_chunk.hip) against the recurrences row by row in 64 bits: the delta
rule with one decay a head and the linear scan with either kind of decay (the rule with a decay a channel has tests of its own)."""
import numpy as np
import pytest
import torch

from plain_ditazen import delta_scan
from plain_novosun import decayed_outer_scan

DEV = "cuda:0"


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(torch.float32).to(DEV)


def ints(a):
    return torch.tensor(list(a), dtype=torch.int32, device=DEV)


@pytest.mark.gpu
@pytest.mark.parametrize("law, heads, share, R, C", [
    ("delta", 4, 2, 128, 128), ("delta", 3, 1, 20, 13), ("delta", 2, 2, 256, 33), ("channel", 3, 1, 128, 80), ("channel", 2, 1, 5, 3),
    ("channel", 2, 2, 200, 17), ("head", 6, 6, 128, 64), ("head", 4, 2, 16, 65), ("head", 1, 1, 77, 16)])
def test_chunks_against_the_recurrence_row_by_row(law, heads, share, R, C):
    """Segments of none, one, fifteen, sixteen, seventeen rows and several chunks, in slabs that cut them, from states that are
    not zero; some decays are zero; work space and results hold NaN before.  The bound is that of the scans row by row."""
    from runtime.kernels import ops
    rng = np.random.default_rng(R + C)
    counts, slots = [17, 0, 1, 83, 15, 16], [3, 6, 0, 5, 1, 4]
    T, starts = sum(counts), np.concatenate(([0], np.cumsum(counts)))
    vec, is_delta = law == "channel", law == "delta"
    groups = heads // share
    q, k, v = (rng.standard_normal((T, n, d)) for n, d in ((groups, R), (groups, R), (heads, C)))
    k /= np.sqrt((k * k).sum(-1, keepdims=True))
    g = rng.uniform(0.6, 1.0, (T, heads, R if vec else 1))
    g[rng.random(g.shape) < 0.02] = 0.0
    b = rng.standard_normal((T, heads)) * 2 if is_delta else rng.uniform(0.1, 2.0, (T, heads))
    begun = rng.standard_normal((7, heads, R, C))
    state = torch.full((7, heads * R * C + 3), 9.0, device=DEV)
    state[:, :heads * R * C] = dev(begun.reshape(7, -1))
    out = torch.full((T, heads * C), float("nan"), device=DEV)
    wide = torch.full((T, groups * R * 2 + 5), 7.0, device=DEV)                     # (q and k as columns of wider rows)
    wide[:, 1:1 + groups * R], wide[:, 2 + groups * R:2 + 2 * groups * R] = dev(q.reshape(T, -1)), dev(k.reshape(T, -1))
    operands = (wide[:, 1:1 + groups * R], wide[:, 2 + groups * R:2 + 2 * groups * R], dev(v.reshape(T, -1)), dev(g.reshape(T, -1)))
    work = torch.full((ops.channel_chunk_work(T, len(counts), heads, R, C, slab=5, delta=is_delta),), float("nan"), device=DEV)
    sizes, kw = (state, ints(starts), ints(slots), heads, R, C, work), dict(share=share, q_scale=0.37, slab=5)
    if is_delta:
        ops.channel_delta_chunks(*operands, dev(b), out, *sizes, **kw)
    else:
        ops.linear_chunks(*operands, out, *sizes, step=None if vec else dev(b), **kw)
    got, after = out.cpu().numpy().reshape(T, heads, C), state.cpu().numpy()
    for s, slot in enumerate(slots):
        rows = slice(starts[s], starts[s + 1])
        for h in range(heads):
            S = begun[slot, h]
            for t in range(rows.start, rows.stop):
                kk, qq, dd = k[t, h // share], q[t, h // share], np.broadcast_to(g[t, h], (R,))
                S = dd[:, None] * S
                u = (v[t, h] - S.T @ kk) / (1.0 + np.exp(-b[t, h])) if is_delta else v[t, h] * (1.0 if vec else b[t, h])
                S = S + np.outer(kk, u)
                want = 0.37 * (S.T @ qq)
                assert np.abs(got[t, h] - want).max() < 2e-5 * max(1.0, np.abs(want).max()), (s, t, h)
            mine = after[slot, h * R * C:(h + 1) * R * C].reshape(R, C)
            assert np.abs(mine - S).max() < 2e-5 * np.abs(S).max(), (s, h)
    assert (after[:, heads * R * C:] == 9.0).all() and np.array_equal(after[[2, 6], :-3], begun[[2, 6]].reshape(2, -1).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("law, heads, share, R, C", [("delta", 4, 2, 128, 128), ("delta", 2, 1, 64, 64), ("channel", 2, 1, 128, 128), ("head", 8, 8, 128, 64)])
@pytest.mark.parametrize("decays", ["near one", "0.8 to one", "any"])
def test_chunks_are_no_further_from_64_bits_than_the_walk_row_by_row(law, heads, share, R, C, decays):
    """The same operands through both forms, 300 rows from a state that is not zero.  Results: the relative error of the chunks is at
    most that of the rows.  The state: within a tenth of it (under strong decays both round a state's last rows a few times,
    and which of the two ends closer depends on the draw)."""
    from runtime.kernels import ops
    T, vec, is_delta = 300, law == "channel", law == "delta"
    gen = torch.Generator(device=DEV).manual_seed(R + C + heads)
    draw = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    unit = lambda x: torch.nn.functional.normalize(x, dim=-1).reshape(T, -1).contiguous()
    q, k, v = unit(draw(T, heads // share, R)), unit(draw(T, heads // share, R)), draw(T, heads * C)
    u = torch.rand(T, heads * R if vec else heads, device=DEV, generator=gen)
    g = {"near one": 1 - 1e-3 * u, "0.8 to one": 0.8 + 0.2 * u, "any": u ** 3}[decays]
    b = draw(T, heads) if is_delta else draw(T, heads).abs() + 0.1
    begun = 0.3 * draw(1, heads * R * C)
    S, want = begun.double().view(heads, R, C), []
    for t in range(T):
        kk, qq = (x[t].double().view(-1, R).repeat_interleave(share, 0) for x in (k, q))
        S = S * g[t].double().view(heads, -1, 1)
        w = v[t].double().view(heads, C)
        w = torch.sigmoid(b[t].double())[:, None] * (w - (S * kk[:, :, None]).sum(1)) if is_delta else w if vec else w * b[t].double()[:, None]
        S = S + kk[:, :, None] * w[:, None, :]
        want.append((S * qq[:, :, None]).sum(1).reshape(-1))
    want, end = torch.stack(want), S.reshape(1, -1)
    where, sizes = (ints([0, T]), ints([0])), (heads, R, C)
    errors = []
    for chunks in (False, True):
        state, out = begun.clone(), torch.empty(T, heads * C, device=DEV)
        work = torch.empty(ops.channel_chunk_work(T, 1, *sizes, delta=is_delta), device=DEV)
        if is_delta:
            args = (q, k, v, g, b, out, state, *where, *sizes)
            ops.channel_delta_chunks(*args, work, share=share) if chunks else ops.delta_scan(*args, share=share)
        else:
            args, kw = (q, k, v, g, out, state, *where, *sizes), dict(share=share, step=None if vec else b)
            ops.linear_chunks(*args, work, **kw) if chunks else ops.linear_scan(*args, **kw)
        errors.append([((x.double() - y).norm() / y.norm()).item() for x, y in ((out, want), (state, end))])
    (rows_out, rows_state), (out, state) = errors
    assert out <= rows_out and state <= 1.1 * rows_state, errors


@pytest.mark.gpu
@pytest.mark.parametrize("is_delta, vec", [(True, False), (True, True), (False, False), (False, True)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_rows_do_not_see_what_is_not_finite_behind_them(is_delta, vec, value):
    """A value, key, query or decay of row 22 (in the middle of a chunk) that is no finite number: the rows before it are what they
    are without it, and so are the other columns where a value holds it."""
    from runtime.kernels import ops
    T, heads, R, C = 40, 2, 32, 32
    gen = torch.Generator(device=DEV).manual_seed(5)
    draw = lambda *shape: torch.randn(*shape, device=DEV, generator=gen)
    q, k, v = draw(T, heads * R) / 6, draw(T, heads * R) / 6, draw(T, heads * C)
    g, b = 0.9 + 0.1 * torch.rand(T, heads * R if vec else heads, device=DEV, generator=gen), draw(T, heads)
    begun = draw(1, heads * R * C)

    def run(q, k, v, g):
        state, out = begun.clone(), torch.empty(T, heads * C, device=DEV)
        work = torch.empty(ops.channel_chunk_work(T, 1, heads, R, C, delta=is_delta), device=DEV)
        where = (out, state, ints([0, T]), ints([0]), heads, R, C, work)
        if is_delta:
            ops.channel_delta_chunks(q, k, v, g, b, *where)
        else:
            ops.linear_chunks(q, k, v, g, *where)
        return out

    want = run(q, k, v, g)
    for which in range(4):
        operands = [q.clone(), k.clone(), v.clone(), g.clone()]
        operands[which][22, 0] = value
        got = run(*operands)
        assert (got[:22] - want[:22]).abs().max().item() < 1e-5 * want.abs().max().item(), which
        if which == 2:
            assert (got[:, 1:] - want[:, 1:]).abs().max().item() < 1e-5 * want.abs().max().item() and not got[22, 0].isfinite()


def test_the_oracle_is_the_designs_recurrence():
    """The loop above is the designs' plain recurrences (from a state of zero, for one head)."""
    rng = np.random.default_rng(1)
    q, k, v, g, b = rng.standard_normal((9, 4)), rng.standard_normal((9, 4)), rng.standard_normal((9, 3)), rng.uniform(0.5, 1, (9, 1)), rng.uniform(0.1, 0.9, 9)
    for is_delta in (True, False):
        S, out = np.zeros((4, 3)), []
        for t in range(9):
            S = g[t][:, None] * S
            S = S + np.outer(k[t], b[t] * (v[t] - S.T @ k[t]) if is_delta else v[t])
            out.append(S.T @ q[t])
        want = delta_scan(q, k, v, b, g[:, 0]) if is_delta else decayed_outer_scan(q, k, v, np.repeat(g, 4, 1))
        np.testing.assert_allclose(out, want, rtol=1e-10, atol=1e-12)


# row by row, by chunks: us on an MI355X of (portions) at (law, heads, rows, columns of a state)
BATCHES = [[48], [2048], [32] * 8, [256] * 8, [1] * 24 + [64], [1] * 64 + [64], [1] * 64 + [512]]
MEASURED = {
    ("delta", 32, 128, 128): [(26, 18), (840, 175), (37, 53), (222, 185), (83, 114), (103, 267), (488, 307)],
    ("delta", 16, 128, 128): [(24, 18), (788, 146), (25, 33), (144, 99), (63, 66), (81, 146), (435, 172)],
    ("channel", 8, 128, 256): [(38, 22), (1401, 107), (37, 33), (244, 84), (76, 60), (101, 123), (492, 140)],
    ("head", 64, 128, 64): [(40, 15), (1392, 161), (44, 48), (274, 197), (91, 100), (130, 235), (532, 280)],
    ("head", 16, 64, 129): [(32, 12), (1178, 83), (31, 23), (212, 70), (58, 40), (71, 87), (402, 100)]}


@pytest.mark.parametrize("law, heads, R, C", MEASURED)
def test_the_form_chosen_is_the_faster_one(law, heads, R, C):
    """Portions alone and beside single rows: what the rule picks takes at most a tenth longer than the other form was measured to."""
    from runtime.engine.context import Batch
    from runtime.parts.recurrent import DeltaByChunks, LinearByChunks
    rule = DeltaByChunks(heads, R, C) if law == "delta" else LinearByChunks(heads, R, C, vector=law == "channel")
    for counts, times in zip(BATCHES, MEASURED[law, heads, R, C]):
        picked = rule.launch_value(Batch(counts, [0] * len(counts), None, False, {}))
        assert times[picked] <= 1.1 * min(times), counts
    assert rule.launch_value(Batch([1] * 9, [5] * 9, None, True, {})) == rule.launch_value(Batch([2] * 64, [0] * 64, None, False, {})) == 0


def test_every_mixer_of_these_laws_names_its_rule():
    """The rule's answer is part of a captured program's key from the first step on."""
    from runtime.parts.recurrent import DeltaByChunks, GatedDeltaRule, GatedLinearAttention, LinearByChunks, MatrixMemory, StateSpaceDuality
    assert GatedDeltaRule("n", 64, 4, 2, 16, 24, 4, 1e-5).step_arrays() == [DeltaByChunks(4, 16, 24)]
    assert GatedLinearAttention("n", 64, 2, 16, 24, 16.0, 1e-5).step_arrays() == [LinearByChunks(2, 16, 24, vector=True)]
    assert StateSpaceDuality("n", 64, 4, 16, 24, 2, 4, 1, 1e-5).step_arrays() == [LinearByChunks(4, 24, 16)]
    assert MatrixMemory("n", 64, 2, 16, 24, 15.0, 1e-5).step_arrays() == [LinearByChunks(2, 16, 25)]


def test_which_steps_walk_the_delta_rule_by_chunks():
    from runtime.engine.context import Batch
    from runtime.parts.recurrent import DeltaByChunks
    value = lambda heads, counts: DeltaByChunks(heads).launch_value(Batch(counts, [0] * len(counts), None, all(n == 1 for n in counts), {}))
    assert value(32, [2048]) == value(32, [1] * 37 + [1024]) == value(16, [256] * 8) == 1
    assert value(32, [1] * 64) == value(32, [20]) == value(32, [32] * 8) == value(16, [64] * 32) == 0
    assert DeltaByChunks(32).words(100, 3) == 0
