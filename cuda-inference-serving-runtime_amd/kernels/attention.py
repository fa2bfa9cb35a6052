"""Paged attention as one call: which kernel, in which form and launch shape, and the step metadata it wants.

`paged_attention` is what a mixer calls.  bfloat16 with a head size in steps of 8 and pages of a power of two >= 8
runs on the matrix cores (one block per row for decode steps, tiles of rows from a task list otherwise); everything
else runs the exact row-wise kernel.  The rules that pick a form or a launch shape are plain functions of sizes
(`rows_launch`, `prompt_form`, `rowwise_splits`), each settled by measurements on an MI355X that its comments quote;
what may be tuned sits in `AttentionTuning`.

The kernels read two kinds of per-step lists that only this file knows the meaning of: task lists (tiles of rows
of one segment) and the rows of the one-token segments of a mixed step.  Both are `StepArray`s: a mixer asks the
step's context for them (`ctx.step_array`), and the step function carries them in every step's metadata from then
on without knowing what they hold.  The reference has one attention kernel and no such choice
(kernels/ops.cu:35-80).
"""
import functools
import math
from dataclasses import dataclass, field
from typing import Optional

import numpy as np
import torch

from . import ops


@dataclass
class AttentionTuning:
    """What the rules below may be told instead of deciding by size (None: decide)."""
    block_tiles: Optional[int] = None     # long portions through LDS-shared tiles of 64 x this items
    square_tiles: Optional[int] = None    # long portions of long contexts through 32 x 32 tiles, 64 x this items a block (0: never)
    square_halves: Optional[int] = None   # two halves a block in that form (even and odd steps): 1, 2
    deep_tiles: Optional[bool] = None     # portions with heads of more than 128 coordinates through LDS-shared tiles of 64 items
    tile_waves: int = 4                   # wavefronts that share one tile's keys
    item_tiles: int = 2                   # 16-item tiles a wave of long portions (small heads)
    # In a mixed step a decoded token is a tile whose keys one block walks; from about this context on the one-token
    # segments get a launch of their own instead, which splits their keys over blocks (SingleRows, single_rows)
    split_single_from: int = 4096
    rows_launch: Optional[tuple] = None   # (wavefronts a block, blocks along the keys) of decode rows
    stream_loads: Optional[bool] = None   # decode rows, and single rows in the square form, read with non-temporal loads (None: by the rules)
    # A step of single tokens whose keys are not split runs a block for every (row, key head), the key heads of a row
    # side by side.  From this many blocks on (more than one block a compute unit) the rows are listed longest first,
    # so that the launch does not end with the blocks of a long row alone (64 rows of 228 to 2,304 keys at the 1.7B
    # sizes: 126.6 -> 119.7 us, what 64 rows of their mean length take; 128 rows at the 135M sizes 36.3 -> 34.2)
    order_rows_from: int = 320


DEFAULT_TUNING = AttentionTuning()


# -- step metadata ----------------------------------------------------------------------------------------------

def fill_tasks(tasks, counts, rows_per_tile, starts=None, skip_single=False):
    """Write (segment, first row, rows, p) for tiles of at most `rows_per_tile` consecutive
    rows of one segment into the int32 array tasks[n, 4]; returns how many were written.
    With `starts` (the position of each segment's first row) p is the position of the tile's
    first row plus one (a segment's rows have consecutive positions, so a kernel that reads p need
    not wait for the positions array; p = 0 says "not given"), and the tiles are ordered by the
    number of keys they attend to, most first: blocks are handed out in this order, and the
    long ones must not be the last to start.  `skip_single`: segments of one row get no tile
    (they are attended to by a launch of their own)."""
    counts = np.asarray(counts, dtype=np.int64)
    tiles = -(-counts // rows_per_tile)
    if skip_single:
        tiles[counts == 1] = 0
    n = int(tiles.sum())
    seg = np.repeat(np.arange(len(counts)), tiles)
    firsts = (np.arange(n) - np.repeat(np.cumsum(tiles) - tiles, tiles)) * rows_per_tile
    made = np.zeros((n, 4), dtype=np.int64)
    made[:, 0] = seg
    made[:, 1] = (np.cumsum(counts) - counts)[seg] + firsts
    made[:, 2] = np.minimum(rows_per_tile, counts[seg] - firsts)
    if starts is not None:
        made[:, 3] = np.asarray(starts, dtype=np.int64)[seg] + firsts + 1
        made = made[np.argsort(-(made[:, 3] + made[:, 2]), kind="stable")]
    tasks[:n] = made
    return n


@dataclass(frozen=True)
class SingleRows:
    """Step array: the rows of the one-token segments of a mixed step (then -1), when they get an attention launch
    of their own: all of them, if one of them has a context of `split_from` keys or more; none in a step of
    one-token segments only, or of short contexts.  Its launch value is how many entries such a launch covers.
    `layer` = (heads, key heads, head size, whether it is one of large heads without a window): `split_from` is multiplied (`least`) where the rows'
    blocks fill the GPU without being split, or run long beside the portions'.  Layers that share a list go by the first one's.
    us together / apart, rows of so many keys beside a portion:
    from 192 blocks and 24 rows on twice: 24 of 4,100 and 64, 32 heads of 128 over 8 (192 blocks) 77 / 96, of 8,000 and 1,024 177 / 196; 64 of
    8,000 and 64, 9 heads over 3, 74 / 75; but with 72 blocks, 24 of 8,000 and 64, 55 / 42, with 24 (16 heads of 256 over one) 227 / 67;
    from 64 blocks on in the square form one and a half times: 24 of 4,100 and 1,024, 9 heads of 64 over 3, 32 / 40, of 8,000 55 / 52.
    Large heads count half (single_rows): 16 of 256 over one, 8 of 2,000 and 64 50 / 23, of 3,000 and 512 73 / 45, of 1,000 and 512 30 / 41;
    but from twice that on (the whole `split_from` of other layers) where the portions take as long as such rows: 400 blocks (8 of 3,000 and 2,048
    105 / 121, of 4,100 138 / 124), or 64 beside as many of single rows (8 of 192 over 2, 40 of 2,000 and 1,024 58 / 76, of 4,100 112 / 108),
    and from a quarter more beside deep tiles (8 of 2,000 and 1,024 63 / 67, of 3,000 87 / 71)."""
    split_from: int
    layer: Optional[tuple] = field(default=None, compare=False)

    def words(self, rows, segments):
        return segments

    def least(self, singles, batch):
        """The context from which on `singles` one-token segments of this batch have a launch of their own."""
        if self.layer is None:
            return self.split_from * (2 if singles >= 24 else 1)
        heads, kv_heads, head_dim, large = self.layer
        group = heads // kv_heads
        chunks = kv_heads * -(-group // min(group, 16))
        unit = 2 * self.split_from if large else self.split_from
        if singles * chunks >= 192:
            return unit * (2 if singles >= 24 else 1)
        if not large and (singles < 24 or singles * chunks < 64):
            return unit
        rows, longest = sum(batch.counts), max(start + count for start, count in zip(batch.starts, batch.counts))
        kind, _, _ = prompt_form(rows, len(batch.counts), 1 << (longest - 1).bit_length(), heads, kv_heads, head_dim, 16, singles=singles)
        if not large:
            return unit * 3 // 2 if kind == "square" else unit
        blocks = -(-(rows - singles) // (64 // min(group, 16))) * chunks
        if singles * chunks >= 64 and blocks >= 64 or blocks >= 400:
            return unit
        return unit * 5 // 8 if kind == "deep" else unit // 2

    def launch_value(self, batch):
        if batch.decode_only or max(batch.starts) + 1 < self.split_from:
            return 0
        singles = [start + 1 for start, count in zip(batch.starts, batch.counts) if count == 1]
        if not singles or max(singles) < self.split_from or max(singles) < self.least(len(singles), batch):
            return 0
        return len(singles)

    def fill(self, out, batch, value):
        out[:] = -1
        if value:
            own = [int(batch.first_row[s]) for s, c in enumerate(batch.counts) if c == 1]
            out[:len(own)] = own


@dataclass(frozen=True)
class SingleTokens:
    """Step array without contents whose launch value is the number of one-token segments in a step that has portions
    too, otherwise 0: what picks a mixed step's form is its portions and how many blocks the others bring (prompt_form)."""

    def words(self, rows, segments):
        return 0

    def launch_value(self, batch):
        return 0 if batch.decode_only else batch.counts.count(1)

    def fill(self, out, batch, value):
        pass


@dataclass(frozen=True)
class RowsLongestFirst:
    """Step array: the rows of a step of one-token segments by the number of keys they attend to, most first (rows of
    equal length in their own order), then the padding rows (which have no keys: zeros are written for them).  Blocks
    are handed out in this order."""

    def words(self, rows, segments):
        return rows

    def launch_value(self, batch):
        return None

    def fill(self, out, batch, value):
        out[:] = np.arange(len(out))
        if batch.decode_only:
            order = np.argsort(-np.asarray(batch.starts, dtype=np.int64), kind="stable")
            out[:len(order)] = np.asarray(batch.first_row, dtype=np.int64)[order]


@functools.lru_cache(maxsize=1024)      # (rules of sizes alone, asked for again in every step's metadata)
def _pieces_launch(pieces, rows, span):
    if pieces.seen:
        span = min(span, pieces.seen)
    blocks = rows * pieces.chunks
    waves, splits = rows_launch(blocks, span, pieces.heads_per_chunk, pieces.head_dim)
    room = rows_room(blocks, span, waves, splits, pieces.head_dim)
    if pieces.merges and splits > 1 and fused_merge_splits(splits, rows, lambda n: ops.merged_rows_ok(rows, pieces.merges, n)) is not None:
        room = None                   # (the product behind merges the rows itself, and those are cut alike)
    if room is None:
        return None, 0.0
    return (room[0], max(rows, -(-room[1] // pieces.chunks)), room[2], splits), rows_even(blocks, span, waves, splits, pieces.head_dim)


@dataclass(frozen=True)
class RowPieces:
    """Step array: how the blocks of a decode step are dealt to its rows by the 32-key steps that each has to walk: int32 [rows +
    1], the first block of every row (rows that pad a step have none) and the end.  Which launch that is for follows from rows
    and the longest context, rounded up to a power of two (`launch`): where a row's keys are not cut the array stays empty.
    Its launch value says whether the step's rows differ enough for that (rows_even): where they do not, it stays empty too, and
    every row's keys are cut alike.  `chunks`: blocks a row and part has; `seen`: how many keys a row sees at most (0: all);
    `merges`: what the product behind can merge itself (ops.merges_into; None: nothing)."""
    chunks: int
    heads_per_chunk: int
    head_dim: int
    window: int
    seen: int
    merges: Optional[tuple] = None

    def launch(self, rows, longest):
        """(wavefronts a block, blocks a key head, least steps a wave, nominal splits) of `rows` rows up to `longest` keys, or None."""
        return _pieces_launch(self, rows, max(256, 1 << (int(longest) - 1).bit_length()))[0]

    def words(self, rows, segments):
        return rows + 1

    def launch_value(self, batch):
        if not batch.decode_only:
            return 0
        longest, n = max(batch.starts) + 1, len(batch.counts)
        rows = batch.rows or n
        even = _pieces_launch(self, rows, max(256, 1 << (longest - 1).bit_length()))[1]
        if even is None:              # (whole rows: the blocks of the rows that there are, dealt to 256 compute units)
            blocks = n * self.chunks
            if blocks <= 0.85 * 256 * -(-blocks // 256):
                return 1
            even = 0.66 if rows * self.chunks <= 512 else 0.0
        if even in (0.0, 1.0):
            return int(even)
        keys, seen = sum(batch.starts) + n, self.seen
        if seen and longest > seen:
            longest, keys = seen, sum([start + 1 if start < seen else seen for start in batch.starts])
        return int(keys <= even * rows * longest)

    def fill(self, out, batch, value):
        """A part is a multiple of the block's waves in steps (each wave then walks as many), the smallest for which the parts of all
        rows are no more than there are blocks; a row has at most 16, or 32 where rows are few and a wave has two steps and
        more (their merge costs more than a second step)."""
        rows = len(out) - 1
        launch = self.launch(rows, max(batch.starts) + 1) if batch.decode_only and value != 0 else None
        if launch is None:
            out[:] = 0
            return
        waves, blocks, a_wave, _ = launch
        ends = np.array(batch.starts) + 1
        steps = ends + 31
        if self.window:
            steps -= np.maximum(ends - self.window, 0) & ~31
        steps >>= 5
        a_wave = max(a_wave, -(-int(steps.sum()) // (waves * blocks)))
        if a_wave == 1 and int(steps.max()) > 32 * waves:
            a_wave = 2                # (more than sixteen parts of two steps a wave instead of sixteen longer ones)
        while True:
            ends = np.minimum((steps + (waves * a_wave - 1)) // (waves * a_wave), 32 if rows < 16 and a_wave > 1 else 16).cumsum()
            if ends[-1] <= blocks:
                break
            a_wave += max(1, a_wave // 8)
        out[0] = 0
        out[1:len(ends) + 1] = ends
        out[len(ends) + 1:] = ends[-1]


@dataclass(frozen=True)
class TileTasks:
    """Step array: the task list of tiles of at most `rows_per_tile` rows, int32 [n, 4]; tiles of no segment
    (-1, 0, 0, 0) pad it.  `singles`: the SingleRows whose launch takes the one-token segments away from the tiles."""
    rows_per_tile: int
    singles: Optional[SingleRows] = None

    def words(self, rows, segments):
        return 4 * (-(-rows // self.rows_per_tile) + segments)   # the most tiles that `rows` rows in `segments` segments make

    def launch_value(self, batch):
        return None

    def fill(self, out, batch, value):
        tasks = out.reshape(-1, 4)
        if batch.decode_only:      # one tile of one row a segment
            n = len(batch.counts)
            tasks[:n, 0] = tasks[:n, 1] = batch.first_row
            tasks[:n, 2] = 1
            tasks[:n, 3] = 0
        else:
            # (layers whose single rows leave the launch by different rules mostly decide alike: one list for both is made once)
            skip = self.singles is not None and batch.launch_values.get(self.singles, 0) > 0
            made = batch.made.get((self.rows_per_tile, skip))
            if made is not None and len(made) == len(out):
                out[:] = made
                return
            n = fill_tasks(tasks, batch.counts, self.rows_per_tile, batch.starts, skip_single=skip)
            batch.made[self.rows_per_tile, skip] = out
        tasks[n:] = (-1, 0, 0, 0)


# -- rules ------------------------------------------------------------------------------------------------------

def prompt_form(rows, n_segments, span, heads, kv_heads, head_dim, page_size, tuning=DEFAULT_TUNING, singles=0):
    """Which form of the matrix-core kernel the prompt rows of a step take, (kind, n, halves): ("tiles", n, 1): a block
    is one tile of 16 n items (a token row and a query head) whose waves split its keys; ("block", n, 1): 64 n items,
    four waves that own different rows and share keys and values through LDS; ("square", n, halves): 64 n items on
    the 32 x 32 instruction with waves of their own for the copies, as one half or as two that take the even and the
    odd steps; ("deep", 1, 1): "block" for heads of more than 128 coordinates.  `span`: the longest context of the step.
    `singles`: how many of the segments are single tokens that share the launch; the others' rows decide, with the singles' blocks counted
    beside theirs (but how large a tile is follows from all rows: a single row is a tile too.  9 heads of 64 over 3, 16 rows of 900 keys
    beside 256, us with 32 items / 16: 11.5 / 9.2, of 3,000 22.8 / 18.5; 8 of 900 beside 1,024 13.9 / 15.8)."""
    tile_items = 2 if tuning.item_tiles == 2 and head_dim <= 64 and rows >= 16 * n_segments else 1
    rows, n_segments = max(1, rows - singles), max(1, n_segments - singles)
    group = heads // kv_heads
    heads_per_chunk = min(group, 16)
    long_portions = rows >= 16 * n_segments
    if singles and head_dim <= 128 and page_size >= 8 and (long_portions or singles >= n_segments) and tuning.square_tiles is None:
        # Decoded tokens beside portions: a block of the square form gives all its waves to a tile of one row, and the
        # single rows' reads run beside the portions' products.  Small blocks (64 items, four waves) leave the compute units room
        # for both; two halves where all the blocks are few and long.  us, before (a single row walked by one wave of a tile) -> now,
        # with 128 items in brackets: 32 heads of 64, 37 rows of 900 keys and a portion of 1,024: 123 -> 74 (82); 30 of
        # 1,300 and one of 30: 99 -> 61 (61); 16 of 200 and one of 256: 22 -> 16 (18); 32 heads of 128 over 8: 78 -> 60
        # (67), 68 -> 44 in halves (46), 22 -> 16 (18).  Below 256 blocks the forms of few blocks below stay ahead (9 heads
        # over 3, 16 of 200 and 256: 11.8 against 13.0), and tiles where the portions are small (fewer than 128 blocks of 64 items; us in this
        # form / in tiles: 32 heads of 64, 8 rows of 900 and a portion of 30 20 / 15, of 100 20 / 16; 32 of 128 over 8, 20 of
        # 2,000 and 30 45 / 37; 8 of 128, 30 of 900 and 256 34 / 29), unless the single rows are more blocks than
        # compute units and their contexts not short (32 heads of 64, 16 of 900 and 30: 25 / 26, of 200 12 / 10).  With large heads larger blocks are ahead where a row's chain
        # of steps is long (30 of 2,400 and 1,024: 98 against 85 with 128 items) or the portions fill the GPU (8 of 2,000 and 2,048: 82
        # against 73 with 192; beside fewer than 192 blocks of single rows from 512 blocks on: 8 of 2,000 and 1,024 41 / 33, 16 of
        # 2,000 48 / 42, but 24 53 / 63).
        # In halves: 30 of 200 and 2,048, 9 heads over 3, 30 / 24, of 2,000 31 / 28; 8 of 128, 16 of 900 and 2,048 46 / 38; with 256
        # blocks of single rows and more they lose (8 of 128, 30 of 900 and 256: 27 / 35).
        chunks = kv_heads * -(-group // heads_per_chunk)
        blocks = -(-rows // (64 // heads_per_chunk)) * chunks
        alone = singles * chunks
        fill = blocks + alone >= 256 and (blocks >= 128 or (alone > 256 and span >= 512))
        if fill and (head_dim <= 64 or (span <= 2048 and blocks < (1000 if alone >= 192 else 512))):
            few = alone < 256 and (blocks + alone <= 384 or (blocks <= 320 and blocks + alone <= 512))
            return "square", 1, 2 if few and span >= 1024 else 1
    if long_portions and head_dim <= 128:
        # enough long portions to fill the GPU with blocks of 64 items (or more): the waves of a block own different
        # rows and share each step's keys and values through LDS.  Otherwise (few heads, short portions) the waves
        # of a block share one tile of 16 items (32 with small heads) and split its keys, which is what hides
        # the latency of a step when blocks are scarce.
        blocks = -(-rows // (64 // heads_per_chunk)) * kv_heads * -(-group // heads_per_chunk)
        # Long contexts: the 32 x 32 form, with three steps in flight a wave.  It costs about 3 us more to start
        # than the others, so it is for tiles that walk a thousand keys and more; larger blocks share the copies
        # among more waves but need more blocks to fill the GPU (MI355X, 2,048 rows: 1.7B sizes 61 us -> 46,
        # 8B sizes 115 -> 71, 135M sizes 32 -> 30; 4,096 rows at the 1.7B sizes: 147 with 128 items, 125 with 256).
        if page_size >= 8 and tuning.square_tiles != 0:
            n = 0
            if tuning.square_tiles is not None:
                n = tuning.square_tiles
            elif span >= 1024 and blocks >= 512:
                # from 2,048 blocks of 64 items on: 192 items, six computing waves beside the two that copy (eight waves:
                # a compute unit holds two such blocks with small heads, one with large, and no wave slot stays empty).
                # 32 heads of 64 at 16k rows: 1.42 ms against 1.46 with 256 items and 1.54 with 128; 9 heads over 3 at
                # 32k: 1.49 against 1.58 and 1.61; 32 heads of 128 over 8 at 8k: 0.60 against 0.63 with 128 items
                # (heads of more than 64 coordinates, one computing wave a SIMD: already from 1,100 blocks on; 32 heads
                # of 128 over 8 at 3,072 rows, 1,536 blocks: 106 us against 123; 24 heads of 96 over 8: 72 against 84)
                n = 3 if blocks >= (2048 if head_dim <= 64 else 1100) else 2
            elif span >= 1024 and blocks >= 128:
                # (fewer blocks than compute units and a thousand keys: 64-item blocks, in two halves; 1,024 rows of
                # 12 heads of 128 take 25 us against 35 as LDS block tiles, of 16 heads of 64 over 4: 17 against 18)
                n = 1
            if n:
                # about one block a compute unit: the time is the longest tile's chain of steps, which two halves a
                # block cut in two (2,048 rows at the 135M sizes 31.6 -> 28.4 us, 4,096 rows 64 -> 55; with more
                # blocks than that the halves only crowd the compute units: 46 -> 68 us at the 1.7B sizes)
                # (up to 511 blocks of 64 items when the chain is long: 3,072 rows at the 135M sizes, 441 blocks,
                # 35.6 us against 43.4; 16 heads over 4 at 1,536 rows 22.1 against 25.4; at 1,000 rows the halves lose)
                # and up to 512 blocks of 128 items from 3,072 keys on: 8 heads of 64 at 6,144 rows 71 against 89,
                # 9 over 3 at 6,144 rows 76 against 92, 16 over 4 at 3,072 rows 42 against 50
                few = (-(-blocks // n) <= 320 or (n == 1 and span >= 1536)
                       or (n == 2 and -(-blocks // n) <= 512 and span >= 3072))
                fits = n == 1 or (n == 2 and head_dim <= 64)
                halves = 2 if (few and fits if tuning.square_halves is None else tuning.square_halves == 2 and fits) else 1
                return "square", n, halves
        block_tiles = (2 if blocks >= 2048 else 1 if blocks >= 512 else 0) if tuning.block_tiles is None else tuning.block_tiles
        if block_tiles:
            return "block", block_tiles, 1
    if long_portions and head_dim > 128 and page_size >= 8:
        # Large heads: the block of 64 items takes 1.4 us a step, a tile's four waves 0.8 (each step's keys straight from the
        # caches, for 16 items).  It is ahead once the tiles wait for the caches: us as tiles / deep, 16 heads of 256 over one key
        # head, 1,000 rows (250 blocks) 91 / 50, 700 and 1,300 rows 186 / 72, 4,096 rows 811 / 282; 8 heads of 192 over 2, 2,048 rows
        # (256 blocks) 107 / 75.  At 128 blocks it depends on the chain: 512 rows of 16 heads over one 40 / 29, 256 rows of 24 heads
        # of 160 over one 25 / 14, the same rows behind 3,000 keys 75 / 106.
        blocks = -(-rows // (64 // heads_per_chunk)) * kv_heads * -(-group // heads_per_chunk)
        if blocks >= (96 if span <= 512 else 192) if tuning.deep_tiles is None else tuning.deep_tiles:
            return "deep", 1, 1
    return "tiles", tile_items, 1


def rows_per_tile_of(form, heads, kv_heads):
    """Rows of one segment that a tile of `form` (prompt_form) holds."""
    kind, n, _ = form
    return (16 if kind == "tiles" else 64) * n // min(heads // kv_heads, 16)


def rowwise_splits(waves, span):
    """Row-wise kernel: how many ways a row's keys are split among wavefronts: enough to
    fill the GPU when the batch alone does not, never finer than 256 keys a split."""
    if waves >= 2048 or span <= 256:
        return 1
    return int(min(32, -(-span // 256), max(1, 4096 // waves)))


def f32_splits(blocks, span):
    """Blocks that share a tile's keys in the float matrix-instruction kernel: until there is a block for every compute unit,
    each of whose eight waves keeps three 16-key steps (a merge costs what two steps take)."""
    return int(max(1, min(256 // max(blocks, 1), span // 384, 32)))


def f32_waves(blocks, span, head_dim):
    """Wavefronts of a block of that kernel.  A compute unit holds two blocks of eight, and where there are more and contexts are
    short most of their waves have no step: from 384 blocks on, up to 512 keys, four, or two with heads of 128 coordinates and from
    768 blocks on.  Single rows, us of 8 / 4 / 2 waves (row by row): 32 heads of 64, 64 rows of 16 keys 21.5 / 11.2 / 9.7 (10.0), of 256
    60 / 44 / 48 (87); 9 heads over 3, 128 rows of 64 keys 7.8 / 6.4 / 8.4 (14.8); 32 heads of 128 over 8, 64 rows of 64 keys 12.8 /
    14.4 / 12.0 (41).  (At 8 keys row by row stays ahead of any: 8.0 against 9.5 us for the 64 rows.)"""
    if blocks < 384 or span > 512:
        return 8
    return 4 if blocks < 768 and head_dim < 128 else 2


def rows_launch(blocks, span, heads_per_chunk, head_dim):
    """Matrix-core decode kernel: (wavefronts a block, blocks along the keys).  Few rows:
    eight waves share a row's keys inside one block; when that still leaves the GPU idle
    and the context is long, the keys are also split over blocks (a merge kernel follows).
    Many rows: four waves a block, one block a row and head group, or with small heads eight waves
    when that gives every compute unit at most one block."""
    steps = -(-span // 32)
    few = blocks < 128
    # eight waves a block with few rows and small heads (at 8k and 32k too: 4 rows at 8k 15.3 us against 16.3 with
    # four waves, 8 rows at 32k 44.4 against 46.5)
    waves = 8 if few and head_dim <= 64 else 4
    if steps <= 2 * waves:
        # two steps a wave: nothing to split (a second block along the keys and the merge cost 2 us of 8 to 10)
        return waves, 1
    if few:
        # Few rows: split the keys until the blocks fill the GPU once: an eight-wave block fills a compute
        # unit (256 blocks; more start a second round: 16 splits of 8 rows at 2k to 4k are 10 % slower than
        # 8), four-wave blocks fit three a unit, of which two are worth having (512 blocks: a thousand are
        # 12 % slower at 30k, where each then lives for three steps a wave only).  A wave keeps at least one
        # 32-key step (with two, 8 rows at 2k have 4 splits and are 5 % slower).
        # At most 32 splits: a single row of 8 key heads at 8k takes 23 us with 32 and 30 with 64.
        room = 256 if waves == 8 else 512
        splits = int(max(1, min(steps // waves, room // blocks, 32)))
        if splits > 16 and steps < 2 * waves * splits:
            # more than 16 splits only with two steps a wave and more: their merge costs more than a second step (one
            # and four rows at 8k keys of the 135M sizes: decode steps of 0.829 and 0.901 ms with 31 and 21 splits,
            # 0.796 and 0.877 with 16; at 32k 32 and 21 splits stay, 16 would take 1.33 against 1.02 ms)
            splits = max(16, steps // (2 * waves))
    elif head_dim <= 64 and 140 <= blocks <= 256:
        # enough rows to give most compute units one block of eight waves, and no more than one each: the
        # keys are not split and no merge follows (9-11 % faster than four waves and three or four splits at
        # 144 to 256 blocks and 2k keys, 4-5 % at 8k)
        waves, splits = 8, 1
    else:
        # Many rows split until every compute unit has the blocks of four waves that its registers hold (three
        # with small heads, two otherwise: 3-5 % faster at 384 blocks of the 135M sizes than one block a unit;
        # from 512 blocks on a split costs 3-8 %); a wave keeps at least four 32-key steps (with two, 128 rows at
        # 512 keys take 19.4 us against 16.5 unsplit).
        target = 768 if head_dim <= 64 else 512
        per = target // blocks if head_dim <= 64 and blocks > 256 else -(-target // blocks)
        splits = int(max(1, min(steps // (waves * 4), per, 64)))
    if waves == 8 and blocks >= 48 and span >= (16384 if blocks < 96 else 6144):
        # Eight-wave blocks whose waves walk long runs of keys: four waves and more blocks along the keys instead, about
        # 1,536 in all, which read with non-temporal loads (`rows_stream_loads`).  Decode steps of the 135M sizes: 32
        # rows at 8k keys 1.865 -> 1.779 ms, 64 rows 2.798 -> 2.755; at 32k 16, 32 and 64 rows 2.695 -> 2.625, 4.713 ->
        # 4.455 and 8.539 -> 8.107; 16 rows at 8k gain nothing.
        waves, splits = 4, int(min(max(1, 1536 // blocks), 16, max(1, steps // 16)))
    return waves, splits


def rows_room(blocks, span, waves, splits, head_dim):
    """Whether a decode step that `rows_launch` gives (waves, splits) deals its blocks to the rows by their lengths, and how:
    (wavefronts a block, blocks that the launch has room for, least 32-key steps a wave), or None: unsplit.
    The launch is filled once: 512 blocks of four waves (256 with more than 128 coordinates, where a compute unit holds one),
    256 of eight, 768 of four with small heads, twice where runs are long.  us of a step of rows between 0.4 and 1.6 times a mean, equal
    splits -> by pieces: 32 heads of 128 over 8, 12 rows of 5,000 keys 76 -> 53, 24 of 3,000 93 -> 62, one of 30,000
    among eight of 500 125 -> 40; 9 of 64 over 3, 100 rows of 1,500 37 -> 30, 64 of 7,000 75 -> 65, 64 of 24,000 239 -> 196; one key head of 256, 24 rows of 2,000
    44 -> 24.  Small heads of many rows that are not split otherwise may be, from 4,096 keys on (below, whole rows longest first are ahead: 32 heads
    of 64, 16 of 1,000 29.2 against 31.9, 64 of 1,216 109 against 114), and so they are with large heads (64 rows of 1,500, 32 heads of 128
    over 8: 71 against 78)."""
    if splits == 1:
        return (4, 1536, 2) if head_dim <= 64 and span >= 4096 and 256 < blocks <= 1024 else None
    if head_dim > 64:
        return 4, (512 if head_dim <= 128 else 256), (1 if blocks < 128 else 2)
    if waves == 8:
        return 8, 256, 1
    return (4, 1536, 4) if blocks * splits > 768 else (4, 768, 2)


def rows_even(blocks, span, waves, splits, head_dim):
    """How even the rows of a decode step may be for its blocks to be dealt by lengths: the most that their keys are of as many rows (the
    padding ones too) of the longest one's length; 1: always, 0: never, None: for whole rows, which RowPieces decides.  Equal rows gain nothing
    and pay for a merge that looks their parts up.  us equal splits / by pieces, that share in brackets: 9 heads of 64 over 3, 32 rows of 9,000
    keys 43.9 / 46.3 (1.0), 45.7 / 47.2 (0.84), 51 / 48.5 (0.63); 64 of 8,000 72 / 73.4 (1.0), 85 / 75.6 (0.63); 12 heads of 64, 32 of 5,000 94.8 /
    101.7 (0.72), 100.4 / 99 (0.63); 32 of 128 over 8, 4 of 3,000 17.7 / 19.3 (1.0), 18.1 / 19.5 (0.87), 20.9 / 20.2 (0.69), 12 of 5,000 and four that
    pad 60.1 / 52.3 (0.75).  Never where a wave has a step at most, and nothing is to be evened out (16 of 128 over 4, 8 of 1,000 12.0 / 13.1 (0.66)).
    Always with more than 16 splits, whose merge by one loop takes longer than the pieces' (32 of 128 over 8, one of 8,000 18.2 / 16.3;
    with more than 128 coordinates only there and where rows differ: 16 of 256 over one, 8 of 6,000 21.4 / 22.5 (1.0), 23.2 / 22.3 (0.74)); where
    the waves' second turn is nearly empty (33 steps of a window for 32 waves: 15.8 / 14.7); and with more than 128 coordinates and more
    blocks than compute units (32 of 1,500 24.7 / 21.8 (1.0), but 16 of 1,500 14.6 / 16.8).  Blocks of eight waves otherwise never
    (12 heads of 64, 8 of 3,000 24.1 / 29.0 (0.74)).
    Whole rows (small heads): where the blocks of the rows that there are leave compute units a sixth idle or more (32 heads of 64, 12 rows of
    5,000 101.6 / 87.1, 20 of 4,500 139 / 126; but 16 of 2,100 50 / 53, 24 of 4,500 147 / 149, 32 of 4,500 193 / 196 and of mixed lengths 196 / 218), or,
    up to 512 blocks, lengths differ much (16 of 4,500 103 / 107 (0.84), 112 / 104 (0.64))."""
    if splits == 1:
        return None
    turns = -(-span // 32) / (waves * splits)
    if head_dim > 128 and blocks * splits > 256:
        return 1.0
    if turns <= 1:
        return 0.0
    if math.ceil(turns) >= 1.3 * turns or (head_dim <= 128 and splits > 16):
        return 1.0
    if head_dim > 128:
        return 0.76 if splits > 16 else 0.0
    return 0.76 if head_dim > 64 else 0.715 if waves == 4 else 0.0


def row_pieces(heads, kv_heads, head_dim, window, keep_first=0, merges=None):
    """The RowPieces of an attention layer."""
    group = heads // kv_heads
    per_chunk = min(group, 16)
    window = int(window or 0)
    return RowPieces(kv_heads * -(-group // per_chunk), per_chunk, head_dim, window, window + 31 + keep_first if window else 0, merges)


def step_arrays(tuning, operand, *layer, law="softmax"):
    """The step arrays that an attention layer names beforehand: what its steps read, as the numbers among them are part of a captured program's key.
    `operand`: one of its matrices (these lists are for the matrix cores, and so for bfloat16); `layer`: what `row_pieces` takes (and
    paged_attention is given); `law`: as in `kernel_units`."""
    heads, kv_heads, head_dim, window = layer[:4]
    if operand is not None and not kernel_units(head_dim, operand.dtype):
        return []
    tokens = [] if law == "sigmoid" else [SingleTokens()]
    pieces = [row_pieces(*layer)] if operand is not None and tuning.rows_launch is None else []
    return [single_rows(tuning, heads, kv_heads, head_dim, window)] + tokens + [RowsLongestFirst()] + pieces


def single_rows(tuning, heads, kv_heads, head_dim, window):
    """The SingleRows of an attention layer.  (Of large heads without a window: half the context.  A window's keys are walked soon.)"""
    large = head_dim > 128 and not window
    return SingleRows(tuning.split_single_from // (2 if large else 1), (heads, kv_heads, head_dim, large))


def rows_stream_loads(blocks, span, waves, splits, head_dim):
    """Whether the decode kernel launched as `blocks` x `splits` blocks of `waves` wavefronts reads keys and values with
    non-temporal loads (no block reads them again; the caches then do not keep them).  Measured inside decode steps
    of the three sizes at 448 to 32,000 keys and 1 to 64 rows: blocks of four waves never lose by them and gain up to
    11 % of the whole step (64 rows at 8k keys of the 8B sizes 4.64 -> 4.12 ms, 32 rows at 2k of the 1.7B sizes 1.379 ->
    1.275).  Blocks of eight waves (head sizes up to 64) gain 2-3 % of the step where they fill the GPU and a wave has
    little more than two 32-key steps (8 and 16 rows at 2k of the 135M sizes, 4 rows at 8k), and lose 2-11 % where a
    wave walks a longer run of keys (four steps and more: 32 and 64 rows at 2k to 32k) or the blocks are few (+4-6 %
    below 96 blocks)."""
    if head_dim > 64 or waves == 4:               # (larger heads run eight waves as four)
        return True
    steps = -(-span // 32)
    return blocks * splits >= 160 and 2 * steps <= 5 * waves * splits


def single_rows_stream(blocks):
    """Whether the single rows of a mixed step in the square form, `blocks` blocks of them (the step's number rounded up), read keys
    and values with non-temporal loads.  The waves' loads take half lines; few blocks leave the caches room to hold a line until its other half is
    asked for, many do not.  us non-temporal / plain: 32 heads of 128 over 8, 8 rows of 4,000 keys and a portion of 256 71 / 60, 8 of 2,000
    and 1,024 50 / 48, 16 of 3,000 and 256 63 / 58, 30 of 900 and 256 30 / 33, 30 of 2,000 and 2,048 107 / 117; 9 heads of 64 over 3,
    8 of 4,000 and 1,024 34 / 23, 50 of 3,000 and 1,024 35 / 31; 32 heads of 64, 3 of 3,000 and 256 30 / 26, 8 of 900 and 30 20 / 21, 30 of 3,000
    and 256 128 / 136.  Where the number is rounded up to 256 the line is crossed early: 20 of 2,000 and 256, 32 heads of 128 over 8, 46 / 38;
    and below it the one place found where plain loads lose is halves beside about a block a compute unit (8 heads of 128, 16 of 900 and 1,024 23 / 26)."""
    return blocks >= 256 or blocks == 0      # (none: one kernel for the portions of all steps)


def fused_merge_splits(splits, rows, accepts):
    """How many of the `splits` blocks along a decode row's keys the product that follows may merge itself
    (`accepts(n)` says whether it takes n), or None: then the merge kernel runs.  That product merges 2, 4 or 8
    partial results of a row while it prepares its operand: one kernel fewer than merging here.  Every block of it
    reads them all, so more than 8 rows bring at most 4 each.  (135M sizes, 8 rows at 2k: a step of 0.808 ms with the
    merge kernel, 0.808 with 4 splits merged there, whose attention blocks are half as many, 0.784 with 8.)  It is
    taken only where it costs at most half of the blocks that `rows_launch` asked for: one row at 8k to 32k keeps its
    24 to 32 splits and the merge kernel."""
    for n in (8, 4, 2):
        if n <= splits and splits <= 2 * n and (n <= 4 or rows <= 8) and accepts(n):
            return n
    return None


# -- the call ---------------------------------------------------------------------------------------------------

def kernel_units(head_dim, dtype, law="softmax"):
    """Names of the shared objects that attention with this head size needs beside the core (library.ensure).
    `law` "sigmoid": the build with sigmoid weights that are not normed over the keys; "distance": the one whose scores
    fall with the distance."""
    from . import library
    if dtype == torch.bfloat16 and head_dim % 8 == 0 and 0 < head_dim <= 256:
        return [library.attention_unit(-(-head_dim // 32) * 32, law)]
    return []


def _split_workspace(ctx, rows, heads, splits, head_dim, dtype=torch.float32, tag="attn.part_o"):
    return (ctx.buffer(tag, (rows * heads * splits * head_dim,), dtype),
            ctx.buffer("attn.part_ml", (rows * heads * splits * 2,), torch.float32))


GATED = "gated"       # paged_attention: the heads' results were packed and gated by the merge


def paged_attention(ctx, q, q_row_stride, kcache, vcache, view, out, heads, kv_heads, head_dim, window, scale,
                    defer_merge=None, tuning=DEFAULT_TUNING, head_bias=None, slopes=None, sink=None, keep_first=0, merge_gate=None, merges=None):
    """out[r] = attention of row r's queries over its request's cached keys up to its own position (or the last
    `window` of them).  `ctx` is the step's context (rows, segments, positions, buffers, step arrays), `view` the
    cache group as the step sees it (block tables, page size).

    `head_bias` (float [heads]): the sigmoid law: a visible key weighs sigmoid(score + head_bias[head]) and the weights
    are not normed over the keys.  Same kernels, launch rules and step arrays, except that prompt rows always run as
    tiles (the forms through LDS have no such build) and no later product merges split keys.
    `slopes` (float [heads]): slopes[head] times the distance is taken off a score; `keep_first`: that many first keys are
    seen besides the window; `sink` (float [heads]): a score that joins the denominator and has no value.

    `defer_merge(splits) -> bool`: the caller's next product can merge the partial results of a decode step whose
    keys are split over `splits` blocks itself (ops.gemm_merged).  Where that is so, no merge kernel runs, `out`
    is left alone and (partial outputs bf16, statistics float, splits) is returned; otherwise None.
    `merges`: what that product's weights are (ops.merges_into), as the layer told `step_arrays`.

    `merge_gate` = (gates, packed, vdim): where the keys of a decode step are split, the merge packs and gates the heads
    itself (ops.attention_mfma) and GATED is returned; otherwise `out` is written and the caller gates."""
    rows = out.shape[0]
    keep_first = int(keep_first) if window else 0
    span = ctx.span_hint if not window else min(ctx.span_hint, window + 31 + keep_first)
    law = dict(head_bias=head_bias, slopes=slopes, sink=sink, keep_first=keep_first)
    common = (q, q_row_stride, kcache, vcache, view.tables, ctx.seg_of_row, ctx.positions, out, heads, kv_heads, head_dim,
              view.page_size, window, scale)
    if (head_bias is None and slopes is None and sink is None and not keep_first
            and ops.attention_f32_ok(q, q_row_stride, kcache, vcache, head_dim, view.page_size)):
        tasks, _ = ctx.step_array(TileTasks(16 // min(heads // kv_heads, 16)))
        tasks = tasks.view(-1, 4)
        blocks = (rows if ctx.decode_only else tasks.shape[0]) * kv_heads * -(-(heads // kv_heads) // 16)
        splits = f32_splits(blocks, span)
        workspace = _split_workspace(ctx, rows, heads, splits, head_dim) if splits > 1 else None
        ops.attention_f32(q, q_row_stride, kcache, vcache, view.tables, ctx.positions, tasks, out, heads, kv_heads, head_dim, view.page_size,
                          window, scale, splits, workspace, f32_waves(blocks, span, head_dim))
        return None
    if not ops.mfma_attention_supported(out.dtype, head_dim, view.page_size):
        splits = rowwise_splits(rows * heads, span)
        workspace = _split_workspace(ctx, rows, heads, splits, head_dim) if splits > 1 else None
        ops.attention_rowwise(*common, splits, workspace, **law)
        return None
    group = heads // kv_heads
    heads_per_chunk = min(group, 16)
    chunks = kv_heads * -(-group // heads_per_chunk)

    def stream(blocks, waves, splits):
        if tuning.stream_loads is not None:
            return tuning.stream_loads
        return rows_stream_loads(blocks, span, waves, splits, head_dim)

    if ctx.decode_only:
        waves, splits = tuning.rows_launch or rows_launch(rows * chunks, span, heads_per_chunk, head_dim)
        if splits > 1 and defer_merge is not None and head_bias is None:
            fused = fused_merge_splits(splits, rows, defer_merge)
            if fused is not None:
                workspace = _split_workspace(ctx, rows, heads, fused, head_dim, torch.bfloat16, "attn.part_o16")
                ops.attention_mfma(*common, None, fused, workspace, waves, merge=False,
                                   stream_loads=stream(rows * chunks, waves, fused), **law)
                return workspace[0], workspace[1], fused
        pieces = row_pieces(heads, kv_heads, head_dim, window, keep_first, merges)
        launch = pieces.launch(rows, ctx.span_hint) if tuning.rows_launch is None else None
        firsts, dealt = ctx.step_array(pieces) if launch is not None else (None, 0)
        if dealt:
            waves, blocks, _, nominal = launch
            ops.attention_mfma(*common, waves=waves, workspace=_split_workspace(ctx, blocks, heads, 1, head_dim), merge_gate=merge_gate,
                               pieces=(firsts[:rows + 1], blocks), stream_loads=stream(rows * chunks, waves, nominal), **law)
            return None if merge_gate is None else GATED
        workspace = _split_workspace(ctx, rows, heads, splits, head_dim) if splits > 1 else None
        order = None
        if splits == 1 and rows * chunks >= tuning.order_rows_from:
            order = ctx.step_array(RowsLongestFirst())[0][:rows]
        gated = merge_gate if splits > 1 else None
        ops.attention_mfma(*common, None, splits, workspace, waves, row_ids=order, stream_loads=stream(rows * chunks, waves, splits),
                           merge_gate=gated, **law)
        return None if gated is None else GATED
    singles = single_rows(tuning, heads, kv_heads, head_dim, window)
    apart, n_single = ctx.step_array(singles)
    if n_single:
        # the decoded tokens of this mixed step: a launch of their own that splits their keys
        waves, splits = tuning.rows_launch or rows_launch(n_single * chunks, span, heads_per_chunk, head_dim)
        workspace = _split_workspace(ctx, n_single, heads, splits, head_dim) if splits > 1 else None
        ops.attention_mfma(*common, None, splits, workspace, waves, row_ids=apart[:n_single],
                           stream_loads=stream(n_single * chunks, waves, splits), **law)
    alone = 0
    if n_single:
        form = prompt_form(max(1, rows - n_single), max(1, ctx.n_segments - n_single), span, heads, kv_heads, head_dim, view.page_size, tuning)
    else:
        if head_bias is None:         # (that law's prompt rows run as tiles in any case)
            _, alone = ctx.step_array(SingleTokens())
        form = prompt_form(rows, ctx.n_segments, span, heads, kv_heads, head_dim, view.page_size, tuning, alone)
    if head_bias is not None and form[0] != "tiles":
        form = ("tiles", 2 if tuning.item_tiles == 2 and head_dim <= 64 else 1, 1)
    if (slopes is not None or keep_first) and form[0] in ("block", "deep"):
        # (that law's build has no such tiles)
        form = ("square", form[1], 1) if form[0] == "block" else ("tiles", 1, 1)
    kind, item_tiles, halves = form
    tasks, _ = ctx.step_array(TileTasks(rows_per_tile_of(form, heads, kv_heads), singles))
    stream_single = kind == "square" and (tuning.stream_loads if tuning.stream_loads is not None else single_rows_stream(alone * chunks))
    ops.attention_mfma(*common, tasks.view(-1, 4), waves=tuning.tile_waves, stream_loads=stream_single,
                       block_tiles={"tiles": False, "block": True, "square": 32, "deep": "deep"}[kind], item_tiles=item_tiles, key_groups=halves,
                       **law)
    return None


def talking_units(dtype, heads, kv_heads, vdim, pad):
    """Names of the shared objects that the attention with mixed scores needs beside the core."""
    from . import library
    return [library.TALKING] if ops.talking_tiles_ok(dtype, heads, kv_heads, vdim, pad, 8) else []


def talking_splits(tiles, span):
    """Blocks that share a tile's keys in the tile form of the attention with mixed scores.  A tile is one block of at
    most eight waves with three barriers a 32-key step, so a compute unit wants two or three blocks to have something to
    run while one waits: the keys are split until the launch has a block for every compute unit, each keeping at least
    four steps.  (2,048 rows of 16 heads of 128 over blocks of 1,024 positions, 129 tiles: 326 us unsplit, 190 with two
    blocks a tile, 193 to 203 with three to six, 227 with eight: the sums that the merge reads grow with the split.)"""
    steps = max(1, -(-span // 32))
    return int(max(1, min(-(-256 // max(tiles, 1)), steps // 4, 8)))


def talking_row_splits(rows, span):
    """Blocks that share a row's keys in the exact form of the attention with mixed scores (one block a row otherwise).
    A block takes about 10 us a tile of 64 keys (its loads wait for each other), so steps of few rows give every tile
    a block of its own until the launch has about four blocks a compute unit."""
    tiles = max(1, -(-span // 64))
    return int(max(1, min(1024 // max(rows, 1), tiles, 32)))


def talking_attention(ctx, q, kcache, vcache, view, out, heads, kv_heads, vdim, pad, mix, scale, temp=None, sink=None,
                      window=None, chunk=None, gate=None):
    """out[r] = attention of row r over its request's cached keys where the scores of all heads of a row are mixed
    (`mix` [heads, heads], after `temp`[g] scale) before the softmax, whose denominator holds exp(`sink`[h]) as well; a
    row sees its block of `chunk` positions up to itself (or the last `window` keys, or all); `gate`: the result times
    sigmoid(gate) element by element.  The mix needs every head's score of a (row, key) pair in one place, so these are
    kernels of their own beside the paged attention above: steps with prompt portions in bfloat16 run tiles of 16 rows
    with all their heads on the matrix cores (the task list of the paged attention's tiles serves); steps of single
    tokens, float32 and sizes the tiles do not take run the exact kernel, one block a row."""
    if not ctx.decode_only and ops.talking_tiles_ok(out.dtype, heads, kv_heads, vdim, pad, view.page_size):
        tasks, _ = ctx.step_array(TileTasks(ops.TALKING_TILE_ROWS))
        rows = out.shape[0]
        splits = talking_splits(tasks.numel() // 4, min(ctx.span_hint, chunk or window or ctx.span_hint))
        workspace = None
        if splits > 1:
            workspace = (ctx.buffer("tattn.part_o", (rows * heads * splits * vdim,), torch.float32),
                         ctx.buffer("tattn.part_ml", (rows * heads * splits * 2,), torch.float32))
        ops.attention_talking_tiles(q, kcache, vcache, view.tables, tasks.view(-1, 4), ctx.positions, out, heads, kv_heads, vdim, pad,
                                    view.page_size, mix, scale, temp=temp, sink=sink, window=window, chunk=chunk, gate=gate,
                                    splits=splits, workspace=workspace)
        return out
    rows = out.shape[0]
    splits = talking_row_splits(rows, min(ctx.span_hint, chunk or window or ctx.span_hint))
    workspace = None
    if splits > 1:
        workspace = (ctx.buffer("tattn.part_o", (rows * heads * splits * vdim,), torch.float32),
                     ctx.buffer("tattn.part_ml", (rows * heads * splits * 2,), torch.float32))
    ops.attention_talking(q, q.stride(0), kcache, vcache, view.tables, ctx.seg_of_row, ctx.positions, out, heads, kv_heads, vdim, pad,
                          view.page_size, mix, scale, temp=temp, sink=sink, window=window, chunk=chunk, gate=gate, splits=splits,
                          workspace=workspace)
    return out
