"""Prompt attention with heads of more than 128 coordinates as blocks of 64 items that share keys and values through LDS: at the edges
of its key steps, tiles, pages, windows and head groups, against plain float32 arithmetic over the same pages."""
import math

import pytest
import torch

from runtime.kernels.attention import AttentionTuning, prompt_form

DEV = "cuda:0"


@pytest.mark.parametrize("heads, kv_heads, dim, rows, span, form", [
    (16, 1, 256, 1000, 1024, "deep"),
    (16, 1, 256, 512, 512, "deep"),          # 128 blocks and a short chain
    (16, 1, 256, 512, 1024, "tiles"),        # the same behind more keys
    (8, 2, 192, 2048, 2048, "deep"),
    (2, 2, 256, 4096, 4096, "tiles"),        # 128 blocks
])
def test_form_of_large_heads_at_measured_points(heads, kv_heads, dim, rows, span, form):
    assert prompt_form(rows, 1, span, heads, kv_heads, dim, 16)[0] == form
    assert prompt_form(rows, 1, span, heads, kv_heads, dim, 4)[0] == "tiles"


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, D", [(16, 1, 256), (3, 1, 136), (24, 1, 160), (40, 2, 168), (4, 4, 192), (5, 5, 224), (8, 1, 248)])
def test_deep_tiles_match_plain_arithmetic(heads, kv_heads, D):
    from test_long_attention_gpu import Step, attend, check
    per = 64 // min(heads // kv_heads, 16)
    step = Step([per + 1, 1, 33, 2 * per, 3, 70, 1], [0, 31, 0, 32, 300, 511, 0])
    got, want = attend(step, heads, kv_heads, D, seed=D, tuning=AttentionTuning(deep_tiles=True))
    check(got, want, f"{heads}/{kv_heads}x{D}")


@pytest.mark.gpu
@pytest.mark.parametrize("window, page_size, sink", [(1, 8, None), (33, 16, 0.5), (64, 32, None), (100, 8, -1.0), (None, 64, 2.0)])
def test_deep_tiles_with_windows_pages_and_a_sink(window, page_size, sink):
    """Values of pages that a row must not see hold NaN; a page that the window has passed is gone from the table."""
    from runtime.kernels import ops
    from runtime.kernels.attention import fill_tasks, rows_per_tile_of
    import numpy as np
    heads, kv_heads, D, counts, starts = 6, 2, 200, [50, 1, 90], [130, 77, 0]
    g = torch.Generator(device=DEV).manual_seed(3)
    per = [-(-(s + c) // page_size) for s, c in zip(starts, counts)]
    pages = sum(per) + 2
    K = torch.randn(pages, kv_heads, page_size, D, generator=g, device=DEV).bfloat16()
    V = torch.full((pages, kv_heads, D, page_size), float("nan"), dtype=torch.bfloat16, device=DEV)
    V[0] = 0.0                                             # (page 0 stands for pages that are gone)
    tables = torch.full((3, max(per)), -1, dtype=torch.int32)
    T = sum(counts)
    q = (3 * torch.randn(T, heads * D, generator=g, device=DEV)).bfloat16()
    want = torch.empty(T, heads, D)
    at, row = 1, 0
    for s, (start, count) in enumerate(zip(starts, counts)):
        n = start + count
        ids = list(range(at, at + per[s]))
        at += per[s]
        gone = 0 if window is None else max(0, start + 1 - window) // page_size     # pages that no row of the step sees
        tables[s, gone:per[s]] = torch.tensor(ids[gone:], dtype=torch.int32)
        values = torch.randn(n, kv_heads, D, generator=g, device=DEV).bfloat16()
        for j in range(n):
            V[ids[j // page_size], :, :, j % page_size] = values[j]
        keys = K[ids].permute(0, 2, 1, 3).reshape(-1, kv_heads, D)[:n].double()
        for i in range(count):
            low = 0 if window is None else max(0, start + i + 1 - window)
            k, v = keys[low:start + i + 1], values[low:start + i + 1].double()
            for h in range(heads):
                scores = k[:, h // 3] @ q[row + i].view(heads, D)[h].double() / math.sqrt(D)
                top = scores.max() if sink is None else torch.clamp(scores.max(), min=sink)
                w = torch.exp(scores - top)
                want[row + i, h] = ((w @ v[:, h // 3]) / (w.sum() + (0.0 if sink is None else torch.exp(sink - top)))).cpu()
        row += count
    seg = torch.tensor(np.repeat(np.arange(3), counts), dtype=torch.int32, device=DEV)
    pos = torch.tensor(np.concatenate([np.arange(s, s + c) for s, c in zip(starts, counts)]), dtype=torch.int32, device=DEV)
    rows = rows_per_tile_of(("deep", 1, 1), heads, kv_heads)
    tasks = np.full((-(-T // rows) + 3, 4), 0, np.int32)
    tasks[:, 0] = -1
    fill_tasks(tasks, counts, rows, starts)
    out = torch.full((T, heads * D), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.attention_mfma(q, heads * D, K, V, tables.to(DEV), seg, pos, out, heads, kv_heads, D, page_size, window, 1.0 / math.sqrt(D),
                       torch.from_numpy(tasks).to(DEV), block_tiles="deep",
                       sink=None if sink is None else torch.full((heads,), sink, device=DEV))
    got = out.float().cpu().view(T, heads, D)
    assert torch.isfinite(got).all()
    # weights and outputs round to bfloat16 (2^-9 each)
    assert (got - want).abs().max() < 8e-3 * want.abs().max() and (got - want).norm() < 4e-3 * want.norm()


@pytest.mark.gpu
def test_deep_tiles_are_refused_where_they_do_not_exist():
    from runtime.kernels import ops
    for D, kw in ((128, {}), (256, dict(item_tiles=2)), (256, dict(head_bias=torch.zeros(1, device=DEV))), (256, dict(slopes=torch.zeros(1, device=DEV)))):
        q = torch.zeros(4, D, dtype=torch.bfloat16, device=DEV)
        cache = torch.zeros(1, 1, 16, D, dtype=torch.bfloat16, device=DEV)
        ints = torch.zeros(4, dtype=torch.int32, device=DEV)
        with pytest.raises(ops.KernelError):
            ops.attention_mfma(q, D, cache, cache.view(1, 1, D, 16), ints.view(4, 1), ints, ints, q.clone(), 1, 1, D, 16, None, 1.0,
                               torch.zeros(1, 4, dtype=torch.int32, device=DEV), block_tiles="deep", **kw)


def _microseconds(step, heads, kv_heads, D):
    from runtime.kernels import attention
    from test_long_attention_gpu import View, make_cache
    K, V, tables = make_cache(step, kv_heads, D, 1)
    q = torch.randn(step.n_rows, heads * D, device=DEV).bfloat16()
    out = torch.empty_like(q)
    tuning = AttentionTuning(deep_tiles=True, split_single_from=1 << 30)
    launch = lambda: attention.paged_attention(step, q, heads * D, K, V, View(tables), out, heads, kv_heads, D, None, D ** -0.5, tuning=tuning)
    launch()
    torch.cuda.synchronize()
    best = math.inf
    for _ in range(5):
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        for _ in range(20):
            launch()
        end.record()
        torch.cuda.synchronize()
        best = min(best, begin.elapsed_time(end) * 50)
    return best


@pytest.mark.gpu
def test_all_waves_of_a_block_walk_a_single_rows_keys():
    """Decoded tokens of 2,000 keys run beside a portion of 1,024 rows; walked by one wave of four they take 1.5 times what it does."""
    from test_long_attention_gpu import Step
    alone = _microseconds(Step([1024], [0]), 16, 1, 256)
    assert _microseconds(Step([1] * 8 + [1024], [1999] * 8 + [0]), 16, 1, 256) < 1.35 * alone


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, D, window", [(16, 1, 256, None), (6, 2, 200, None), (3, 3, 160, None), (16, 1, 256, 40), (3, 3, 192, 50)])
def test_deep_tiles_keep_what_is_not_finite_from_other_waves_rows(heads, kv_heads, D, window):
    """Values of some keys hold NaN and infinities.  They reach the rows that see them, and at most the rows that share their sixteen items (with
    16 heads a key head none: a wave's items are one row): not a block's earlier rows, nor those whose window has passed them."""
    from runtime.kernels import attention
    from test_long_attention_gpu import P, Step, View, make_cache
    step, gc = Step([150, 1, 90], [0, 33, 64]), min(heads // kv_heads, 16)
    K, V, tables = make_cache(step, kv_heads, D, 4)
    for s, key, d, what in [(0, 3, 5, math.nan), (0, 17, 40, math.inf), (0, 70, 9, -math.inf), (0, 141, D - 1, math.nan), (1, 33, 0, math.nan), (2, 100, 77, math.inf),
                            (2, 153, 78, math.nan)]:
        V[tables[s, key // P].item(), :, d, key % P] = what
    q = torch.randn(step.n_rows, heads * D, device=DEV).bfloat16()
    out = torch.empty_like(q)
    attention.paged_attention(step, q, heads * D, K, V, View(tables), out, heads, kv_heads, D, window, D ** -0.5, tuning=AttentionTuning(deep_tiles=True))
    got, row, kept = out.double().cpu().view(-1, heads, D), 0, 0
    for s, (start, count) in enumerate(zip(step.starts, step.counts)):
        pages = tables[s, :-(-(start + count) // P)].long()
        keys = K[pages].double().cpu().permute(0, 2, 1, 3).reshape(-1, kv_heads, D)
        values = V[pages].double().cpu().permute(0, 3, 1, 2).reshape(-1, kv_heads, D)
        for i in range(count):
            for h in range(heads):
                at, per = h * kv_heads // heads, 64 // gc
                wave = (i % per * gc + h % gc) // 16
                first, last = (min(i // per * per + item // gc, i // per * per + per - 1, count - 1) for item in (16 * wave, 16 * wave + 15))
                low, near = (0 if window is None else max(0, start + x + 1 - window) for x in (i, first))
                k, v = keys[low:start + i + 1, at], values[low:start + i + 1, at]
                sees, may = ~torch.isfinite(v).all(0), ~torch.isfinite(values[near:start + last + 1, at]).all(0)
                odd = ~torch.isfinite(got[row, h])
                assert (odd >= sees).all() and (odd <= may).all(), (s, i, h)
                want = torch.softmax(k @ q[row].double().cpu().view(heads, D)[h] * D ** -0.5, 0) @ v
                # (a weight as two bf16 numbers and the output's rounding, 2^-9)
                assert (got[row, h] - want)[~odd].abs().max() < 8e-3 * max(1.0, want[~odd].abs().max())
                kept += int((~may).sum())
            row += 1
    assert kept > 0
