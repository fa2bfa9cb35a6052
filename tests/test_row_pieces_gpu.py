"""Decode steps whose blocks are dealt to the rows by their lengths (kernels.attention.RowPieces)."""
import math

import numpy as np
import pytest
import torch

from runtime.engine.context import Batch
from runtime.kernels.attention import RowPieces, row_pieces


@pytest.mark.parametrize("heads, kv_heads, dim, window", [(32, 8, 128, 0), (9, 3, 64, 0), (32, 32, 64, 0), (16, 1, 256, 1024), (16, 4, 128, 1024), (40, 2, 96, 600)])
def test_every_row_gets_its_parts_and_no_more_than_there_are(heads, kv_heads, dim, window):
    rng = np.random.default_rng(heads + window)
    pieces, cut = row_pieces(heads, kv_heads, dim, window), 0
    for n, rows in [(1, 1), (2, 2), (12, 16), (33, 64), (64, 64), (1, 4), (100, 128)] * 3:
        starts = [int(x) for x in np.exp(rng.uniform(0, math.log(60000), n))]
        out = np.full(pieces.words(rows, rows), 7, dtype=np.int32)
        pieces.fill(out, Batch([1] * n, starts, np.arange(n, dtype=np.int32), True, {}), None)
        launch = pieces.launch(rows, max(starts) + 1)
        if launch is None:
            assert (out == 0).all()
            continue
        waves, blocks, least, _ = launch
        parts = np.diff(out)
        assert out[0] == 0 and out[-1] <= blocks and (parts[n:] == 0).all()
        assert (parts[:n] >= 1).all() and parts.max() <= 32
        # what a wave walks is what the mean would give it, rounded up, unless the row has all the parts that it may have
        steps = np.array([(s + 1 - (max(s + 1 - window, 0) & ~31 if window else 0) + 31) // 32 for s in starts])
        a_wave = -(-(-(-steps // parts[:n])) // waves)
        fair = max(least, 2, math.ceil(steps.sum() / (waves * max(1, blocks - n))))
        assert (a_wave[parts[:n] < 16] <= 1.2 * fair + 1).all()
        cut += int((parts > 1).sum())
    assert cut > 20


def test_steps_with_portions_have_no_pieces():
    pieces = row_pieces(32, 8, 128, None)
    out = np.full(pieces.words(40, 3), 7, dtype=np.int32)
    pieces.fill(out, Batch([38, 1, 1], [0, 900, 70], np.array([0, 38, 39], dtype=np.int32), False, {}), None)
    assert (out == 0).all()


@pytest.mark.parametrize("heads, kv_heads, dim, window, lengths, rows, dealt", [
    (9, 3, 64, 0, [8000] * 64, 64, 0),                                  # rows of one length: cut alike
    (9, 3, 64, 0, [4000, 12000] * 32, 64, 1),
    (9, 3, 64, 0, [9000] * 32, 32, 0),
    (9, 3, 64, 0, [8000] * 4, 4, 0),
    (9, 3, 64, 0, [8200] * 4, 4, 1),                                    # 21 splits
    (12, 12, 64, 0, [3000] * 4 + [2000] * 4, 8, 0),                     # blocks of eight waves
    (32, 8, 128, 0, [5000] * 8, 8, 0),
    (32, 8, 128, 0, [5000] * 12, 12, 0),
    (32, 8, 128, 0, [5000] * 12, 16, 1),                                # four rows that pad
    (32, 8, 128, 0, [3000] * 4, 4, 0),
    (32, 8, 128, 0, [700, 300, 200], 4, 0),                             # a step a wave
    (32, 32, 64, 0, [2100] * 16, 16, 0),                                # whole rows: two blocks a compute unit
    (32, 32, 64, 0, [5000] * 12, 16, 1),                                # one and a half
    (32, 32, 64, 0, [6900, 2100] * 8, 16, 1),
    (32, 32, 64, 0, [6900, 2100] * 16, 32, 0),                          # 1,024 blocks: they even out by themselves
    (16, 1, 256, 0, [1500] * 8, 8, 0),
    (16, 1, 256, 0, [1500] * 32, 32, 1),                                # 512 blocks of which a compute unit holds one
    (16, 1, 256, 1024, [1500] * 8, 8, 1),                               # 33 steps for 32 waves
    (16, 4, 128, 1024, [1100] * 24, 32, 1),
])
def test_blocks_are_dealt_by_lengths_where_rows_differ(heads, kv_heads, dim, window, lengths, rows, dealt):
    n, pieces = len(lengths), row_pieces(heads, kv_heads, dim, window)
    batch = Batch([1] * n, [x - 1 for x in lengths], np.arange(n, dtype=np.int32), True, {}, rows)
    assert pieces.launch_value(batch) == dealt
    out = np.full(pieces.words(rows, rows), 7, dtype=np.int32)
    pieces.fill(out, batch, dealt)
    assert (out == 0).all() if not dealt else (out[-1] > n or dealt == 1)
    assert pieces.launch_value(Batch([1, 2], [900, 0], np.array([0, 1], dtype=np.int32), False, {}, 4)) == 0


def test_no_list_is_made_where_the_product_behind_merges():
    """Four rows of 1,000 to 5,000 keys, 32 heads of 128 over 8: the output projection takes the rows' partial results as they are."""
    batch = Batch([1] * 4, [4999, 999, 1999, 999], np.arange(4, dtype=np.int32), True, {}, 4)
    assert row_pieces(32, 8, 128, None).launch_value(batch) == 1
    merged = row_pieces(32, 8, 128, None, merges=(4096, 32, 128))
    out = np.full(5, 7, dtype=np.int32)
    merged.fill(out, batch, None)
    assert merged.launch(4, 5000) is None and merged.launch_value(batch) == 0 and (out == 0).all()
    assert merged.launch(16, 5000) == row_pieces(32, 8, 128, None).launch(16, 5000) is not None        # (more rows than it merges)


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, D, length, law", [(9, 3, 64, 9000, None), (32, 8, 128, 3000, "gate"), (16, 1, 256, 1500, None)])
def test_rows_of_one_length_are_cut_alike(heads, kv_heads, D, length, law):
    """The same call, and the same bits, as with the launch rule's splits given."""
    from runtime.kernels import attention
    from test_long_attention_gpu import DEV, Step, View, make_cache
    n = 4 if D == 128 else 32 if D == 64 else 8
    step = Step([1] * n, [length - 1] * n)
    K, V, tables = make_cache(step, kv_heads, D, seed=1)
    q = (torch.randn(n, heads * D, device=DEV) * 2.0).bfloat16()
    gates, packed = torch.randn(n, heads * D, device=DEV), [torch.zeros(n, heads * D, dtype=torch.bfloat16, device=DEV) for _ in range(2)]
    outs = []
    chunks = kv_heads * -(-(heads // kv_heads) // 16)
    given = attention.rows_launch(n * chunks, step.span_hint, min(heads // kv_heads, 16), D)
    for i, tuning in enumerate((attention.DEFAULT_TUNING, attention.AttentionTuning(rows_launch=given))):
        out = torch.zeros(n, heads * D, dtype=torch.bfloat16, device=DEV)
        left = attention.paged_attention(step, q, heads * D, K, V, View(tables), out, heads, kv_heads, D, None, D ** -0.5, tuning=tuning,
                                         merge_gate=None if law is None else (gates, packed[i], D))
        assert (left == attention.GATED) == (law == "gate")
        outs.append(packed[i] if law else out)
    assert outs[0].any() and torch.equal(*outs)
    assert any(isinstance(a, RowPieces) and not dealt for a, (_, dealt) in step.arrays.items())


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, D, lengths, window, law", [
    (32, 8, 128, [7750, 31, 2300, 5001, 1, 640], None, None),          # groups of 4: pieces of many sizes, a row of one key
    (9, 3, 64, [9000, 500, 33], None, None),                           # eight waves a block
    (32, 16, 64, [3000, 700], 600, None),                              # a window
    (16, 1, 256, [1500, 90, 2047, 800], None, None),                   # large heads
    (40, 2, 96, [4000, 65], None, "sink"),                             # two chunks a key head
    (16, 4, 128, [1100, 40, 1900], 1024, "sigmoid"),                   # plain sums
    (8, 2, 128, [5000, 64, 1300], None, "gate"),                       # packed and gated by the merge
    (8, 2, 64, [5000, 900, 1300], 1024, "slopes"),
])
def test_rows_of_mixed_lengths_by_pieces(monkeypatch, heads, kv_heads, D, lengths, window, law):
    from runtime.kernels import attention
    monkeypatch.setattr(RowPieces, "launch_value", lambda self, batch: 1)           # (also where the rows' lengths are no reason for it)
    from test_long_attention_gpu import DEV, Step, View, make_cache
    n = len(lengths)
    step = Step([1] * n, [x - 1 for x in lengths])
    K, V, tables = make_cache(step, kv_heads, D, seed=heads + D)
    rows = n + 2                                                        # two rows that pad the step
    g = torch.Generator(device=DEV).manual_seed(5)
    q = (torch.randn(rows, heads * D, generator=g, device=DEV) * 2.0).bfloat16()
    bias, vdim = torch.randn(heads, generator=g, device=DEV) - 3.0, D - 40
    slopes = torch.rand(heads, generator=g, device=DEV) * 0.01
    gates = torch.randn(rows, heads * vdim, generator=g, device=DEV)
    step.n_rows = step.n_segments = rows
    step.seg_of_row = torch.cat([step.seg_of_row, torch.full((2,), -1, dtype=torch.int32, device=DEV)])
    step.positions = torch.cat([step.positions, torch.zeros(2, dtype=torch.int32, device=DEV)])
    tables = torch.cat([tables, torch.full((2, tables.shape[1]), -1, dtype=torch.int32, device=DEV)])
    out = torch.full((rows, heads * D), float("nan"), dtype=torch.bfloat16, device=DEV)
    packed = torch.full((rows, heads * vdim), float("nan"), dtype=torch.bfloat16, device=DEV)
    scale = 1.0 / math.sqrt(D)
    extra = {"sink": dict(sink=bias), "sigmoid": dict(head_bias=bias), "gate": dict(merge_gate=(gates, packed, vdim)),
             "slopes": dict(slopes=slopes, keep_first=17)}.get(law, {})
    attention.paged_attention(step, q, heads * D, K, V, View(tables), out, heads, kv_heads, D, window, scale, **extra)
    assert any(isinstance(a, RowPieces) and dealt for a, (_, dealt) in step.arrays.items()), "this step is meant to be dealt by pieces"
    group = heads // kv_heads
    want = torch.zeros(rows, heads, D, dtype=torch.float64, device=DEV)
    for s, length in enumerate(lengths):
        pages = tables[s, :-(-length // 16)].long()
        keys = K[pages].double().permute(1, 0, 2, 3).reshape(kv_heads, -1, D)[:, :length].repeat_interleave(group, 0)
        values = V[pages].double().permute(1, 0, 3, 2).reshape(kv_heads, -1, D)[:, :length].repeat_interleave(group, 0)
        x = (keys * q[s].double().view(heads, 1, D)).sum(-1) * scale                     # [heads, length]
        at = torch.arange(length, device=DEV)
        if law == "slopes":
            x = x - slopes.double()[:, None] * (length - 1 - at)
        seen = at > length - 1 - (window or length) if law != "slopes" else (at > length - 1 - window) | (at < 17)
        if law == "sigmoid":
            w = torch.sigmoid(x + bias.double()[:, None]) * seen
        else:
            x = x.masked_fill(~seen, float("-inf"))
            if law == "sink":
                x = torch.cat([x, bias.double()[:, None]], 1)
            w = torch.softmax(x, -1)[:, :length]
        want[s] = (w[:, :, None] * values).sum(1)
    got = out
    if law == "gate":
        got, want = packed, (want[:, :, :vdim] * torch.sigmoid(gates.double().view(rows, heads, vdim)))
    got, want = got.double().view(rows, -1), want.reshape(rows, -1)
    torch.cuda.synchronize()
    assert torch.isfinite(got).all() and (got[n:] == 0).all()
    # the weights are rounded to bf16 as operands (2^-9 each, independent over the keys) and so is the result (2^-9)
    assert (got - want).norm() < 4e-3 * want.norm()
    assert ((got - want).norm(dim=1)[:n] < 8e-3 * want.norm(dim=1)[:n]).all()
