"""The rules that pick a kernel's form are plain functions of sizes: their decisions at the points where
measurements settled them (profiles/prompt_attention_forms_and_the_rule_that_picks.txt and
profiles/decode_attention_launch_shapes_and_the_rule_that_picks.txt), so that a change of a rule shows."""
import pytest
import torch

from runtime.kernels.attention import fused_merge_splits, prompt_form, rows_launch, rows_stream_loads


@pytest.mark.parametrize("heads, kv_heads, dim, rows, form", [
    (9, 3, 64, 2048, ("square", 1, 2)),       # about one block a compute unit: two halves a block
    (9, 3, 64, 3072, ("square", 1, 2)),       # 441 blocks, a long chain: still halves
    (9, 3, 64, 6144, ("square", 2, 2)),       # 440 blocks of 128 items from 3,072 keys on
    (9, 3, 64, 8192, ("square", 2, 1)),
    (32, 32, 64, 2048, ("square", 2, 1)),
    (32, 32, 64, 4096, ("square", 3, 1)),     # 2,048 blocks of 64 items: 192 items a block
    (32, 8, 128, 2048, ("square", 2, 1)),
    (32, 8, 128, 3072, ("square", 3, 1)),     # large heads: 192 items from 1,100 blocks on
    (16, 4, 64, 3072, ("square", 2, 2)),
    (16, 4, 64, 6144, ("square", 2, 1)),      # 768 blocks of 128 items: the halves would crowd the compute units
])
def test_prompt_attention_form_at_measured_points(heads, kv_heads, dim, rows, form):
    assert tuple(prompt_form(rows, 1, rows, heads, kv_heads, dim, 16)) == form


def test_prompt_attention_form_needs_long_portions_and_pages_of_eight_keys():
    assert prompt_form(40, 8, 3000, 9, 3, 64, 16)[0] == "tiles"        # many short portions
    assert prompt_form(2048, 1, 2048, 9, 3, 64, 4)[0] != "square"      # the copying waves take 8 keys of a page
    assert prompt_form(2048, 1, 2048, 2, 2, 256, 16)[0] == "tiles"     # heads of more than 128 coordinates


@pytest.mark.parametrize("blocks, keys, group, dim, launch", [
    (3, 2048, 3, 64, (8, 8)),          # one request of the 135M sizes
    (24, 2048, 3, 64, (8, 8)),         # eight
    (192, 2048, 3, 64, (8, 1)),        # 64: one block of eight waves a compute unit, no split
    (24, 8192, 3, 64, (8, 10)),        # eight waves at long contexts too
    (3, 8192, 3, 64, (8, 16)),         # one request at 8k: 16 splits of two steps a wave, not 31 of one
    (12, 8192, 3, 64, (8, 16)),
    (3, 32768, 3, 64, (8, 32)),        # at 32k a wave has steps enough for 32 splits
    (12, 32768, 3, 64, (8, 21)),
    (96, 8192, 3, 64, (4, 16)),        # but from 16 rows on four waves and about 1,536 blocks in all (non-temporal loads)
    (192, 32768, 3, 64, (4, 8)),
    (48, 8192, 3, 64, (8, 5)),         # 16 rows at 8k stay
    (48, 32768, 3, 64, (4, 16)),
    (24, 512, 3, 64, (8, 1)),          # two steps a wave: nothing to split
    (384, 512, 3, 64, (4, 1)),
    (8, 8192, 4, 128, (4, 32)),        # at most 32 splits
    (64, 2048, 4, 128, (4, 8)),
    (512, 2048, 4, 128, (4, 1)),
])
def test_decode_attention_launch_at_measured_points(blocks, keys, group, dim, launch):
    assert tuple(rows_launch(blocks, keys, group, dim)) == launch


@pytest.mark.parametrize("blocks, keys, group, dim, streams", [
    (24, 2048, 3, 64, True),           # eight requests of the 135M sizes: 192 blocks of eight waves, one step a wave
    (3, 2048, 3, 64, False),           # one request: few blocks
    (192, 2048, 3, 64, False),         # 64 requests unsplit: a wave walks eight steps
    (24, 8192, 3, 64, False),
    (12, 8192, 3, 64, True),           # 4 requests at 8k: 21 splits, a step and a half a wave
    (2048, 2048, 1, 64, True),         # four waves a block: always
    (8, 8192, 4, 128, True),           # large heads: always
    (512, 512, 4, 128, True),
])
def test_decode_attention_streams_keys_and_values_at_measured_points(blocks, keys, group, dim, streams):
    waves, splits = rows_launch(blocks, keys, group, dim)
    assert rows_stream_loads(blocks, keys, waves, splits, dim) is streams


@pytest.mark.parametrize("splits, rows, fused", [
    (8, 8, 8),         # eight requests of the 135M sizes at 2k: the output projection merges all eight
    (10, 8, 8),        # at 8k the rule asks for ten: eight merged there still beat ten and a merge kernel
    (8, 16, 4),        # more than 8 rows bring at most four each
    (4, 16, 4),
    (32, 1, None),     # one row at 8k to 32k keeps its 32 splits: a quarter of the blocks would cost more than the merge kernel
    (24, 1, None),
    (3, 4, 2),
    (1, 8, None),
])
def test_splits_that_the_output_projection_merges_itself(splits, rows, fused):
    assert fused_merge_splits(splits, rows, lambda n: True) == fused
    assert fused_merge_splits(splits, rows, lambda n: False) is None


@pytest.mark.parametrize("rows, columns, k, ring", [
    (3100, 16384, 2048, True),         # 208 GFLOP with a short inner size: ahead of the library by up to 25 %
    (4096, 16384, 2048, False),
    (640, 28672, 4096, True),
    (777, 28672, 4096, False),         # 183 GFLOP with a long one: the library by 4 to 15 %
    (907, 28672, 4096, False),
    (1500, 16384, 4096, False),
    (500, 36864, 5120, False),
])
def test_ring_product_of_gate_and_up_at_measured_points(rows, columns, k, ring):
    from runtime.kernels import ops
    w = torch.empty(columns, k, dtype=torch.bfloat16, device="meta")
    assert ops.ring_ahead(rows, w, gated=True) is ring


def test_ring_product_of_gate_and_up_where_the_library_takes_no_operands():
    """Rows or weights that are views: the other side is not the library, and the product stays here."""
    from runtime.kernels import ops
    w = torch.empty(28672, 4224, dtype=torch.bfloat16, device="meta")
    assert ops.ring_ahead(777, w[:, :4096], gated=True)
    assert ops.ring_ahead(777, w[:, :4096].contiguous(), gated=True, library_rows=False)


@pytest.mark.parametrize("kind, rows, columns, k, apart", [
    ("gelu", 1280, 8192, 2048, False),
    ("gelu", 1999, 8192, 2048, True),          # 16 M results: 67 us as two kernels, 74 with the epilogue
    ("gelu_tanh", 4096, 4096, 1024, True),
    ("relu2", 1999, 8192, 2048, False),
    ("relu2", 4096, 8192, 2048, True),
    ("gelu", 8000, 2048, 2048, False),         # a narrow product that ends with its store is the ring product's in any case
])
def test_activation_of_a_large_product_at_measured_points(kind, rows, columns, k, apart):
    from runtime.kernels import ops
    half = lambda *shape: torch.empty(*shape, dtype=torch.bfloat16, device="meta")
    a, w, out, product = half(rows, k), half(columns, k), half(rows, columns), half(rows, columns)
    assert ops.activation_apart(a, w, out, product, kind) is apart
    # what only the epilogue takes stays with it: no buffer, results or rows in a view
    assert not ops.activation_apart(a, w, out, None, kind)
    assert not ops.activation_apart(a, w, half(rows, columns + 8)[:, 8:], product, kind)
    assert not ops.activation_apart(half(rows, k + 64)[:, 64:], w, out, product, kind)


@pytest.mark.parametrize("rows, columns, k, floats, ring", [
    (17, 8512, 2048, True, False),         # 33 MB of weights, float results: 11.6 us in the streaming kernel, 12.8 here
    (32, 10240, 2048, True, False),
    (33, 8512, 2048, True, True),
    (17, 49152, 576, True, True),          # 54 MB: 17.8 / 14.4
    (32, 6144, 2048, False, True),         # bf16 results
])
def test_ring_product_of_few_rows_at_measured_points(rows, columns, k, floats, ring):
    from runtime.kernels import ops
    w = torch.empty(columns, k, dtype=torch.bfloat16, device="meta")
    assert ops.ring_ahead(rows, w, floats=floats) is ring


def test_products_that_never_leave_a_norm_are_told_by_their_sizes(monkeypatch):
    """The host asks every product of a pre-norm layer whether it leaves the norm behind it: few rows and wide ones are not planned for."""
    from runtime.kernels import ops
    monkeypatch.setattr(ops, "ring_ahead", lambda *a, **k: pytest.fail("asked further"))
    for rows, cols in ((1, 576), (64, 576), (1061, 1028), (65, 4096)):
        a, w = torch.empty(rows, 64, dtype=torch.bfloat16), torch.empty(cols, 64, dtype=torch.bfloat16)
        assert ops.ring_normed_parts(a, w, torch.empty(rows, cols), torch.empty(cols)) == 0


@pytest.mark.parametrize("rows, weight_rows, k, rope, inside", [
    (1, 3072, 576, False, True), (512, 3072, 576, False, True),            # 31.9 us apart, 29.5 inside
    (640, 3072, 576, False, False), (640, 3072, 768, False, True),         # 37.0 / 39.0, 44.9 / 44.0
    (1024, 3072, 768, False, False), (4096, 8192, 576, False, False),      # 63.0 / 64.5, 438 / 522
    (8, 49152, 576, False, True), (32, 49152, 576, False, True),           # a head: 31.1 / 30.1
    (33, 49152, 576, False, False), (130, 49152, 576, False, False),       # 54 / 63 (40 rows), 122 / 148
    (1, 49152, 256, False, False), (1, 32768, 256, False, True),           # 12.3 / 13.0, 9.6 / 9.2
    (1, 128256, 576, False, False), (1, 128256, 768, False, True),         # 58.3 / 58.5, 86.4 / 81.6
    (2048, 960, 576, True, True), (4096, 960, 576, True, True),            # the rotation behind it: 40.9 / 38.4, 75.5 / 73.1
    (1024, 3072, 576, True, True), (2048, 3072, 576, True, False),         # 58.8 / 58.8
])
def test_where_a_32_bit_product_makes_its_rows_norm(rows, weight_rows, k, rope, inside):
    from runtime.kernels.ops import f32_norm_ahead
    assert f32_norm_ahead(rows, weight_rows, k, rope) is inside
