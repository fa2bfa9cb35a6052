"""Attention of steps that hold decoded tokens beside prompt portions: the rule that picks their form, and single rows inside the
square form (all waves of a block take one row's keys) at the edges of its key steps, pages and head groups."""
import pytest
import torch

from runtime.engine.context import Batch
from runtime.kernels.attention import AttentionTuning, SingleRows, SingleTokens, prompt_form


def test_single_tokens_of_a_step():
    """The launch value counts the one-token segments, and only where portions share the step."""
    def value(counts):
        return SingleTokens().launch_value(Batch(counts, [0] * len(counts), None, all(c == 1 for c in counts), {}))
    assert [value(c) for c in ([1, 5, 1], [1, 5, 9, 2], [5, 9], [7], [1, 1], [1])] == [2, 1, 0, 0, 0, 0]
    assert SingleTokens().words(64, 8) == 0


def test_single_rows_share_the_launch_up_to_twice_the_context_when_they_are_many():
    def value(n, context):
        return SingleRows(100).launch_value(Batch([1] * n + [6], [context - 1] * n + [0], None, False, {}))
    assert [value(23, 99), value(23, 100), value(24, 199), value(24, 200), value(1, 100)] == [0, 23, 0, 24, 1]


def test_layers_name_the_numbers_that_they_read_and_no_others():
    """A step's launch values are part of its captured program's key."""
    from runtime.kernels.attention import DEFAULT_TUNING, RowPieces, RowsLongestFirst, step_arrays

    def named(dtype, head_dim=64, **law):
        return [type(a) for a in step_arrays(DEFAULT_TUNING, torch.zeros(1, 1, dtype=dtype), 8, 2, head_dim, None, **law)]
    assert named(torch.bfloat16) == [SingleRows, SingleTokens, RowsLongestFirst, RowPieces]
    assert named(torch.bfloat16, law="sigmoid") == [SingleRows, RowsLongestFirst, RowPieces]
    assert named(torch.float32) == named(torch.bfloat16, 20) == []          # (row by row, or the 32-bit tiles)


@pytest.mark.parametrize("heads, kv_heads, dim, singles, rows, span, form", [
    (32, 32, 64, 37, 1024, 2048, ("square", 1, 1)),
    (32, 32, 64, 16, 256, 256, ("square", 1, 1)),       # 640 blocks, short contexts
    (32, 8, 128, 16, 256, 1024, ("square", 1, 2)),      # 256 blocks
    (32, 8, 128, 37, 1024, 2048, ("square", 1, 1)),
    (32, 8, 128, 30, 1024, 4096, ("square", 2, 1)),     # large heads, long rows: the portions' own form
    (9, 3, 64, 37, 1024, 2048, ("square", 1, 2)),       # 255 blocks
    (9, 3, 64, 16, 256, 256, ("tiles", 2, 1)),
    (32, 32, 64, 30, 30, 2048, ("square", 1, 1)),
    (32, 32, 256, 30, 300, 2048, ("tiles", 1, 1)),      # 160 blocks
    (32, 32, 256, 30, 400, 2048, ("deep", 1, 1)),
])
def test_form_of_mixed_steps_at_measured_points(heads, kv_heads, dim, singles, rows, span, form):
    assert tuple(prompt_form(rows + singles, 1 + singles, span, heads, kv_heads, dim, 16, singles=singles)) == form
    assert prompt_form(rows + singles, 1 + singles, span, heads, kv_heads, dim, 4, singles=singles)[0] != "square"


@pytest.mark.parametrize("heads, kv_heads, dim, window, singles, portion, least", [
    (16, 1, 256, None, 24, 64, 2048),          # 24 blocks
    (16, 1, 256, None, 40, 1024, 2560),        # deep tiles beside them
    (16, 1, 256, None, 8, 2048, 4096),         # which take longer than the rows
    (16, 1, 256, 1024, 8, 64, 4096),
    (8, 2, 192, None, 40, 1024, 4096),         # 80 blocks beside 128
    (8, 2, 192, None, 40, 64, 2048),
    (32, 32, 256, None, 8, 64, 4096),          # 256 blocks
    (8, 8, 192, None, 24, 256, 8192),          # 192
    (9, 3, 64, None, 24, 64, 4096),            # 72 blocks, tiles
    (9, 3, 64, None, 24, 1024, 6144),          # the square form
    (9, 3, 64, None, 64, 64, 8192),            # 192 blocks
    (9, 3, 64, None, 8, 1024, 4096),
    (32, 8, 128, None, 23, 1024, 4096),
    (32, 8, 128, None, 24, 64, 8192),
])
def test_single_rows_leave_the_launch_by_blocks_and_form(heads, kv_heads, dim, window, singles, portion, least):
    from runtime.kernels.attention import DEFAULT_TUNING, step_arrays
    array = step_arrays(DEFAULT_TUNING, None, heads, kv_heads, dim, window)[0]

    def value(context):
        return array.launch_value(Batch([1] * singles + [portion], [context - 1] * singles + [0], None, False, {}))
    assert (value(least - 1), value(least)) == (0, singles)


@pytest.mark.parametrize("heads, kv_heads, dim, singles, rows, span, form", [
    (9, 3, 64, 16, 256, 1024, ("tiles", 2, 1)),         # 272 rows of 17 segments
    (9, 3, 64, 16, 255, 1024, ("tiles", 1, 1)),         # 271: a single row is a tile of 16 items
    (9, 3, 64, 32, 288, 1024, ("tiles", 1, 1)),
    (9, 3, 64, 32, 2048, 1024, ("square", 1, 2)),       # 294 blocks beside 96: halves
    (8, 8, 128, 16, 2048, 1024, ("square", 1, 2)),
    (8, 8, 128, 32, 2048, 1024, ("square", 1, 1)),      # 256 blocks of single rows
    (32, 32, 64, 8, 56, 1024, ("tiles", 1, 1)),         # a small portion
    (32, 32, 64, 8, 192, 1024, ("tiles", 2, 1)),        # 96 blocks
    (32, 32, 64, 8, 256, 1024, ("square", 1, 1)),
    (32, 32, 64, 16, 48, 256, ("tiles", 1, 1)),         # 512 blocks of single rows, short contexts
    (32, 32, 64, 16, 48, 1024, ("square", 1, 1)),
    (32, 8, 128, 8, 1024, 2048, ("square", 2, 1)),      # 512 blocks beside 64: the portions' own form
    (32, 8, 128, 32, 1024, 2048, ("square", 1, 1)),     # beside 256
])
def test_single_rows_are_no_reason_for_a_slower_form(heads, kv_heads, dim, singles, rows, span, form):
    assert tuple(prompt_form(rows + singles, 1 + singles, span, heads, kv_heads, dim, 16, singles=singles)) == form


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, D", [(9, 3, 64), (32, 8, 128), (4, 4, 32), (20, 1, 96), (6, 2, 72)])
def test_single_rows_in_square_tiles(heads, kv_heads, D):
    """Single rows of 1 to 300 keys (no key but their own, a step less one, a step, one more, a wave's second step) beside portions
    whose last tile is one row too, in every size of block and in halves; then a step that takes the form by the rule."""
    from test_long_attention_gpu import Step, attend, check
    keys = [1, 2, 15, 16, 17, 31, 32, 33, 64, 127, 255, 256, 257, 300]
    per = 64 // min(heads // kv_heads, 16)
    step = Step([1] * 7 + [per + 1] + [1] * 7 + [3, 2 * per + 1], [k - 1 for k in keys[:7]] + [40] + [k - 1 for k in keys[7:]] + [500, 0])
    for n, halves in ((1, 1), (1, 2), (2, 1), (2, 2), (3, 1), (4, 1)):
        if D > 64 and (n == 4 or (n == 2 and halves == 2)):
            continue
        got, want = attend(step, heads, kv_heads, D, seed=n, tuning=AttentionTuning(square_tiles=n, square_halves=halves))
        check(got, want, f"{heads}/{kv_heads}x{D}, blocks of {64 * n} items, {halves} halves")
    step = Step([1] * 90 + [200], [7 * i for i in range(90)] + [100])
    if kv_heads >= 3:
        assert prompt_form(290, 91, step.span_hint, heads, kv_heads, D, 16, singles=90)[0] == "square"
    got, want = attend(step, heads, kv_heads, D, seed=9)
    check(got, want, f"{heads}/{kv_heads}x{D}, 90 single rows and 200")


@pytest.mark.gpu
@pytest.mark.parametrize("heads, kv_heads, D, singles, streams", [(32, 8, 128, 8, False), (32, 8, 128, 32, True), (9, 3, 64, 64, False), (32, 32, 64, 8, True)])
def test_few_single_rows_read_with_plain_loads(monkeypatch, heads, kv_heads, D, singles, streams):
    """Which loads the single rows of the square form take, and that their results do not depend on it."""
    from runtime.kernels import ops
    from test_long_attention_gpu import Step, attend
    step, seen, launch = Step([1] * singles + [1024], [37 * i for i in range(singles)] + [700]), [], ops.attention_mfma
    monkeypatch.setattr(ops, "attention_mfma", lambda *a, **kw: (seen.append((kw.get("block_tiles"), kw.get("stream_loads"))), launch(*a, **kw))[1])
    by_rule, _ = attend(step, heads, kv_heads, D, seed=3)
    assert seen == [(32, streams)]
    for stream in (False, True):
        got, _ = attend(step, heads, kv_heads, D, seed=3, tuning=AttentionTuning(stream_loads=stream))
        assert torch.equal(got, by_rule)
