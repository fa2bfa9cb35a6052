"""The 32-bit path's attention on the float matrix instruction (csrc/attention_f32.hip) against attention row by row in 64 bits."""
import math

import numpy as np
import pytest
import torch

from test_kernels_gpu import DEV, f64, paged_case, reference_attention, rnd, tol

pytestmark = pytest.mark.gpu


def tasks_of(rows, per):
    """Tiles of at most `per` neighbouring rows of one segment, a tile of no segment among them."""
    tasks, at = [(-1, 0, 0, 0)], 0
    while at < len(rows):
        n = 1
        while n < per and at + n < len(rows) and rows[at + n][0] == rows[at][0] and rows[at + n][1] == rows[at][1] + n:
            n += 1
        tasks.append((rows[at][0], at, n, 0))
        at += n
    return torch.tensor(tasks, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("heads, kv_heads, dim, page_size", [(9, 3, 64, 16), (4, 4, 32, 4), (8, 1, 128, 8), (20, 1, 96, 64), (16, 1, 64, 32), (34, 2, 32, 16)])
@pytest.mark.parametrize("window", [None, 1, 9, 40])
def test_attention_f32(heads, kv_heads, dim, page_size, window):
    """Segments of one key to several hundred (more than a turn of the eight waves), tiles of whole prompts and of their ends, single
    rows; groups of heads that fill a tile, leave some of it and take two; windows whose earlier pages are gone; more splits
    than a short segment has keys.  Scores spread by 2.8, so that maxima move: up to about 13, whose rounding (a few of 2^-24 of it) moves a
    weight by up to 3e-6 of itself and a result, values of up to 4, by 1e-5; the row-wise kernel's bound else."""
    from runtime.kernels import ops
    _, kt, vt, tables, _ = paged_case(heads, kv_heads, dim, page_size, [17, 7, 1, 330], torch.float32, seed=dim + heads)
    group = heads // kv_heads
    scale = 0.7 / math.sqrt(dim)
    at = {0: range(10, 17), 1: range(4, 7), 2: [0], 3: [*(() if window else range(5)), 200, *range(290, 330)]}
    rows = [(seg, pos) for seg, where in at.items() for pos in where]
    qt = rnd(len(rows), heads, dim, seed=3, scale=4.0)
    want = reference_attention(qt, kt, vt, tables, rows, page_size, window=window, scale=scale)
    if window:                                             # pages that no row of a segment sees are gone, and hold NaN
        tables = tables.clone()
        for seg in range(tables.shape[0]):
            low = min(pos for s, pos in rows if s == seg) + 1 - window
            for j in range(max(0, low) // page_size):
                kt[tables[seg, j]] = vt[tables[seg, j]] = float("nan")
                tables[seg, j] = -1
    T = len(rows)
    pos = torch.tensor([r[1] for r in rows], dtype=torch.int32, device=DEV)
    tasks = tasks_of(rows, 16 // min(group, 16))
    wide = torch.full((T, heads * dim + 8), float("nan"), device=DEV)
    wide[:, 4:4 + heads * dim] = qt.reshape(T, -1)
    for splits in (1, 3, 33):
        out = torch.full((T, heads * dim), 7.0, device=DEV)
        ws = (torch.full((T * heads * splits * dim,), float("nan"), device=DEV), torch.full((T * heads * splits * 2,), float("nan"), device=DEV))
        ops.attention_f32(wide.view(-1)[4:], wide.stride(0), kt, vt, tables, pos, tasks, out, heads, kv_heads, dim, page_size, window, scale, splits, ws)
        np.testing.assert_allclose(f64(out).reshape(T, heads, dim), want, rtol=tol(torch.float32)["rtol"], atol=1e-5, err_msg=f"splits={splits}")


def test_what_attention_f32_takes():
    from runtime.kernels import ops
    q = torch.zeros(4, 64, device=DEV)
    kc = vc = torch.zeros(2, 1, 16, 64, device=DEV)
    assert ops.attention_f32_ok(q, 64, kc, vc, 64, 16)
    assert not any(ops.attention_f32_ok(q, 64, kc, vc, dim, page) for dim, page in ((48, 16), (256, 16), (64, 2), (64, 12)))
    assert not ops.attention_f32_ok(q.bfloat16(), 64, kc, vc, 64, 16) and not ops.attention_f32_ok(q, 66, kc, vc, 64, 16)
    assert not ops.attention_f32_ok(q.view(-1)[1:], 64, kc, vc, 64, 16)


@pytest.mark.parametrize("heads, kv_heads, dim", [(9, 3, 64), (32, 8, 128), (8, 1, 128), (4, 4, 32)])
def test_no_further_from_64_bits_than_the_row_wise_kernel(heads, kv_heads, dim):
    """Single rows of wide scores (spread 3) at a few hundred keys, where a score's own rounding decides: the relative error is at
    most the row-wise kernel's on the same operands."""
    from runtime.kernels import ops
    lengths, page = [200, 320, 77, 450], 16
    _, kt, vt, tables, _ = paged_case(heads, kv_heads, dim, page, lengths, torch.float32, seed=dim)
    rows = [(s, n - 1) for s, n in enumerate(lengths)]
    q, scale = rnd(len(rows), heads, dim, seed=3, scale=3.0), 1.0 / math.sqrt(dim)
    want = reference_attention(q, kt, vt, tables, rows, page, scale=scale)
    ints = lambda a: torch.tensor(a, dtype=torch.int32, device=DEV)
    pos, flat, errors = ints([p for _, p in rows]), q.reshape(len(rows), -1).contiguous(), []
    for tiles in (False, True):
        out = torch.empty(len(rows), heads * dim, device=DEV)
        args = (out, heads, kv_heads, dim, page, None, scale)
        if tiles:
            ops.attention_f32(flat, heads * dim, kt, vt, tables, pos, tasks_of(rows, 16 // min(heads // kv_heads, 16)), *args)
        else:
            ops.attention_rowwise(flat, heads * dim, kt, vt, tables, ints([s for s, _ in rows]), pos, *args)
        errors.append(np.linalg.norm(f64(out).reshape(want.shape) - want) / np.linalg.norm(want))
    assert errors[1] <= errors[0], errors


@pytest.mark.parametrize("window", [None, 6])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_rows_do_not_see_what_is_not_finite_where_they_do_not_look(window, value):
    """Rows 30 to 45 of a prompt, sixteen a tile, and a value of key 36 that is no finite number: the rows that do not see that key
    are what they are without it, and so are the other coordinates."""
    from runtime.kernels import ops
    heads, dim, page = 2, 32, 16
    _, kt, vt, tables, _ = paged_case(heads, heads, dim, page, [46], torch.float32, seed=1)
    pos = torch.arange(30, 46, dtype=torch.int32, device=DEV)
    q = rnd(16, heads * dim, seed=2)
    tasks, outs = torch.tensor([(0, 0, 16, 0)], dtype=torch.int32, device=DEV), []
    for _ in range(2):
        outs.append(torch.empty(16, heads * dim, device=DEV))
        ops.attention_f32(q, heads * dim, kt, vt, tables, pos, tasks, outs[-1], heads, heads, dim, page, window, dim ** -0.5)
        vt[tables[0, 2], 1, 3, 36 - 32] = value
    want, got = outs
    sees = (pos >= 36) & (pos - 36 < (window or 99))
    assert (got[~sees] - want[~sees]).abs().max().item() < 1e-5 and not got[sees, dim + 3].isfinite().any()
    other = torch.arange(heads * dim, device=DEV) != dim + 3
    assert (got[:, other] - want[:, other]).abs().max().item() < 1e-5


@pytest.mark.parametrize("where", ["query", "key", "value", "scores of -inf"])
def test_what_is_not_finite_reaches_the_rows_that_see_it(where):
    """A query, a key or a value that is no number, and scores that are all -inf, whose weights are none: no number as row by row, in the same
    rows and coordinates."""
    from runtime.kernels import ops
    heads, dim, page, n = 2, 32, 16, 40
    _, kt, vt, tables, _ = paged_case(heads, heads, dim, page, [n], torch.float32, seed=1)
    pos = torch.arange(20, n, dtype=torch.int32, device=DEV)
    q = rnd(n - 20, heads * dim, seed=2)
    if where == "query":
        q[3, 5] = float("nan")
    elif where == "key":
        kt[tables[0, 1], 1, 30 - 16, 7] = float("nan")
    elif where == "value":
        vt[tables[0, 1], 1, 7, 30 - 16] = float("nan")
    else:
        kt[:, 0, :, 0] = -float("inf")
        q[:, 0] = q[:, 0].abs() + 0.1
    tasks, seg = torch.tensor([(0, 0, 16, 0), (0, 16, 4, 0)], dtype=torch.int32, device=DEV), torch.zeros(n - 20, dtype=torch.int32, device=DEV)
    want, args = torch.empty(n - 20, heads * dim, device=DEV), (heads, heads, dim, page, None, dim ** -0.5)
    ops.attention_rowwise(q, heads * dim, kt, vt, tables, seg, pos, want, *args)
    assert want.isnan().any() and not want.isnan().all()
    for waves in (2, 8):
        got = torch.empty(n - 20, heads * dim, device=DEV)
        ops.attention_f32(q, heads * dim, kt, vt, tables, pos, tasks, got, *args, waves=waves)
        assert torch.equal(got.isnan(), want.isnan()) and torch.allclose(got, want, rtol=1e-4, atol=1e-5, equal_nan=True)


@pytest.mark.parametrize("heads, kv_heads, dim", [(9, 3, 64), (4, 4, 32), (8, 1, 128), (6, 2, 96)])
@pytest.mark.parametrize("waves", [2, 4])
def test_attention_f32_with_fewer_waves(heads, kv_heads, dim, waves):
    """Blocks of two and four waves, with no step for some of them and with several for each, whole and with split keys: the result in 64 bits
    (weights as in test_attention_f32), and the bits of eight waves where no wave has a second step."""
    from runtime.kernels import ops
    page, lengths = 16, [1, 16, 17, 16 * waves, 16 * waves + 1, 130]
    _, kt, vt, tables, _ = paged_case(heads, kv_heads, dim, page, lengths, torch.float32, seed=dim)
    rows = [(seg, pos) for seg, n in enumerate(lengths) for pos in range(max(0, n - 7), n)]
    q, scale = rnd(len(rows), heads, dim, seed=4), dim ** -0.5
    want = reference_attention(q, kt, vt, tables, rows, page, scale=scale)
    pos = torch.tensor([r[1] for r in rows], dtype=torch.int32, device=DEV)
    tasks, flat, outs = tasks_of(rows, 16 // min(heads // kv_heads, 16)), q.reshape(len(rows), -1).contiguous(), {}
    for splits, w in ((1, waves), (3, waves), (1, 8)):
        out = torch.full((len(rows), heads * dim), 7.0, device=DEV)
        ws = (torch.empty(len(rows) * heads * splits * dim, device=DEV), torch.empty(len(rows) * heads * splits * 2, device=DEV))
        ops.attention_f32(flat, heads * dim, kt, vt, tables, pos, tasks, out, heads, kv_heads, dim, page, None, scale, splits, ws, w)
        np.testing.assert_allclose(f64(out).reshape(want.shape), want, rtol=tol(torch.float32)["rtol"], atol=1e-5, err_msg=f"splits={splits}")
        outs[splits, w] = out
    short = torch.tensor([lengths[seg] <= 16 * waves for seg, _ in rows], device=DEV)
    assert torch.equal(outs[1, waves][short], outs[1, 8][short])
    with pytest.raises(ops.KernelError):
        ops.attention_f32(flat, heads * dim, kt, vt, tables, pos, tasks, out, heads, kv_heads, dim, page, None, scale, waves=3)


def test_many_blocks_of_short_contexts_have_few_waves():
    from runtime.kernels.attention import f32_waves
    assert [f32_waves(n, 256, 64) for n in (1, 383, 384, 767, 768, 8192)] == [8, 8, 4, 4, 2, 2]
    assert f32_waves(384, 256, 128) == 2 and f32_waves(8192, 513, 64) == f32_waves(383, 16, 128) == 8
