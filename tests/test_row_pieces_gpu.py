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
def test_rows_of_mixed_lengths_by_pieces(heads, kv_heads, D, lengths, window, law):
    from runtime.kernels import attention
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
    assert any(isinstance(a, RowPieces) for a in step.arrays), "this step is meant to be dealt by pieces"
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
