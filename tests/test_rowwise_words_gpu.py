"""The row-wise kernels of the recurrent mixers and the gelu where they run in 16-byte words, at the edges of those forms."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def close(got, want, tol):
    got, want = got.double().cpu(), want.double().cpu()
    assert ((got - want).abs().max() / want.abs().max().clamp_min(1e-30)).item() < tol


def ints(a):
    return torch.tensor([int(x) for x in a], dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("channels, taps, heads, bias", [(4, 2, 0, True), (1028, 4, 3, True), (300, 3, 300, False), (8, 4, 1, False),
                                                         (27000, 2, 0, True), (26004, 4, 3, True), (26500, 3, 300, False)])
def test_short_convolution_in_words(channels, taps, heads, bias):
    """Portions shorter than the taps, of one row, of more rows than a block takes, that begin inside a block and at its first
    row; rows of no segment; inputs and state as columns of wider rows.  Few channels keep a thread an input (the step is too
    small for the form in words), many take the words."""
    from runtime.kernels import ops
    counts, slots = [5, 1, 43, 0, 16, 2, 33], [2, 0, 5, 1, 6, 3, 4]
    pad, T = 3, sum(counts) + 3
    starts = np.concatenate(([0], np.cumsum(counts)))
    seg = np.concatenate([np.repeat(np.arange(len(counts)), counts), [-1] * pad])
    wide = torch.randn(T, 4 + channels + heads + (-(channels + heads) % 4), device=DEV)
    x, dt = wide[:, 4:4 + channels], wide[:, 4 + channels:4 + channels + heads]
    w, b = torch.randn(channels, taps, device=DEV), torch.randn(channels, device=DEV) if bias else None
    state = torch.randn(7, (taps - 1) * channels + 5, device=DEV)
    before, out = state.clone(), torch.full((T, channels), 9.0, device=DEV)
    gates = None
    if heads:
        step, decay = torch.full((T, heads), 9.0, device=DEV), torch.full((T, heads), 9.0, device=DEV)
        dt_bias, a_log = torch.randn(heads, device=DEV), torch.randn(heads, device=DEV)
        gates = (dt, dt_bias, a_log, step, decay)
    ops.conv_silu(x, w, b, state[:, :(taps - 1) * channels], out, ints(seg), ints(starts), ints(slots), gates=gates)
    for s, slot in enumerate(slots):
        lo, hi = starts[s], starts[s + 1]
        old = before[slot, :(taps - 1) * channels].view(taps - 1, channels).double()
        inputs = torch.cat((old, x[lo:hi].double()))
        z = sum(inputs[j:j + hi - lo] * w[:, j].double() for j in range(taps)) + (0.0 if b is None else b.double())
        if hi > lo:
            close(out[lo:hi], torch.nn.functional.silu(z), 2e-6)
            close(state[slot, :(taps - 1) * channels].view(taps - 1, channels), inputs[-(taps - 1):], 1e-9)
        if heads and hi > lo:
            d = torch.nn.functional.softplus(dt[lo:hi].double() + dt_bias.double())
            close(step[lo:hi], d, 2e-6)
            close(decay[lo:hi], torch.exp(-a_log.double().exp() * d), 2e-6)
    assert (out[-pad:] == 9.0).all() and (state[1] == before[1]).all() and (not heads or bool((step[-pad:] == 9.0).all()))


@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("before", [1, 3, 13, 15, 16])
def test_short_convolution_wherever_a_portion_begins(taps, before):
    """A portion of 70 rows behind another one of `before` rows, against the same portion alone: the rows that lie in blocks of its own
    there lie in shared ones here, blocks whose first row is its second or fourth among them.  The same sums, so the same bits."""
    from runtime.kernels import ops
    channels, n = 26004, 70
    x, w, b = torch.randn(before + n, channels, device=DEV), torch.randn(channels, taps, device=DEV), torch.randn(channels, device=DEV)
    kept, outs = torch.randn(2, (taps - 1) * channels, device=DEV), []
    for rows, counts, slots in ((x, [before, n], [1, 0]), (x[before:].contiguous(), [n], [0])):
        out, state = torch.empty_like(rows), kept.clone()
        ops.conv_silu(rows, w, b, state, out, ints(np.repeat(np.arange(len(counts)), counts)), ints(np.cumsum([0] + counts)), ints(slots))
        outs.append((out[-n:], state[0]))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


@pytest.mark.parametrize("taps", [2, 4])
@pytest.mark.parametrize("channels", [26116, 26144, 26172, 26112])
def test_short_convolution_where_few_lanes_are_left(channels, taps):
    """A row's last wave with 1, 8, 15 and all lanes; blocks that begin deep in a portion, in whose first, ninth, middle and last rows the
    next portion or the padding begins.  Against 64 bits, the last channels apart; the padding stays."""
    from runtime.kernels import ops
    counts, pad = [24, 23, 32, 17, 25, 30], 5                   # portions from rows 24, 47, 79, 96, 121 on, padding from row 151
    T, starts = sum(counts) + pad, np.concatenate(([0], np.cumsum(counts)))
    assert [int(s) % 16 for s in starts[1:]] == [8, 15, 15, 0, 9, 7]
    x, w, b = torch.randn(T, channels, device=DEV), torch.randn(channels, taps, device=DEV), torch.randn(channels, device=DEV)
    state = torch.randn(len(counts), (taps - 1) * channels, device=DEV)
    before, out = state.clone(), torch.full((T, channels), 9.0, device=DEV)
    ops.conv_silu(x, w, b, state, out, ints(np.concatenate([np.repeat(np.arange(len(counts)), counts), [-1] * pad])), ints(starts),
                  ints(range(len(counts))))
    for s, n in enumerate(counts):
        lo = int(starts[s])
        inputs = torch.cat((before[s].view(taps - 1, channels).double(), x[lo:lo + n].double()))
        want = torch.nn.functional.silu(sum(inputs[j:j + n] * w[:, j].double() for j in range(taps)) + b.double())
        last = channels // 256 * 256 if channels % 256 else channels - 256
        close(out[lo:lo + n, :last], want[:, :last], 2e-6)
        close(out[lo:lo + n, last:], want[:, last:], 2e-6)
    assert (out[-pad:] == 9.0).all()


@pytest.mark.parametrize("groups, size", [(300, 4), (33, 128), (9, 132), (40, 256), (3, 260), (2, 1000), (1, 1028), (1, 2048), (1, 4096), (5, 100)])
@pytest.mark.parametrize("gate_first, sigmoid, skip, shared, dtype", [(True, False, True, False, torch.bfloat16), (False, True, False, True, torch.float32),
                                                                     (False, False, True, False, torch.bfloat16)])
def test_group_norm_and_gate_in_words(groups, size, gate_first, sigmoid, skip, shared, dtype):
    from runtime.kernels import ops
    rows, width = max(2, -(-259 // groups)), groups * size
    y, w = torch.randn(rows, width, device=DEV), torch.randn(size if shared else width, device=DEV)
    gate, x = torch.randn(rows, width + 8, device=DEV)[:, 4:4 + width], torch.randn(rows, width + 4, device=DEV)[:, :width]
    d = torch.randn(groups, device=DEV)
    out = torch.empty(rows, width, device=DEV, dtype=dtype)
    ops.group_norm_gate(y, gate, w, out, groups, 1e-5, gate_first=gate_first, shared_weight=shared, sigmoid=sigmoid, skip=(d, x) if skip else None)
    u, z = y.double(), gate.double()
    if skip:
        u = u + d.double().repeat_interleave(size) * x.double()
    law = torch.sigmoid(z) * (1.0 if sigmoid else z)
    if gate_first:
        u = u * law
    u = u.view(rows, groups, size)
    u = (u * torch.rsqrt(u.square().mean(-1, keepdim=True) + 1e-5)).view(rows, width) * (w.double().repeat(groups) if shared else w.double())
    close(out, u if gate_first else u * law, 3e-6 if dtype == torch.float32 else 5e-3)


@pytest.mark.parametrize("rows, cols, rank", [(1025, 256, 16), (513, 520, 3), (130, 2049, 17), (3, 100, 5), (2051, 1024, 16), (1033, 700, 40)])
def test_low_rank_decays_several_rows_a_thread(rows, cols, rank):
    from runtime.kernels import ops
    low, up, bias = torch.randn(rows, rank + 3, device=DEV)[:, 1:1 + rank], torch.randn(rank, cols, device=DEV), torch.randn(cols, device=DEV)
    out = ops.decay_gate_low_rank(low, up, bias, torch.empty(rows, cols, device=DEV), 16.0)
    close(out, torch.exp(torch.nn.functional.logsigmoid(low.double() @ up.double() + bias.double()) / 16.0), 2e-6)


@pytest.mark.parametrize("n", [8, 2048 * 8 + 8, 12, (2 << 20) + 8, (2 << 20) + 12])
@pytest.mark.parametrize("form", ["gelu", "gelu_tanh"])
def test_gelu_of_bf16_words(n, form):
    from runtime.kernels import ops
    x = (torch.randn(1, n, device=DEV) * 3).bfloat16()
    out = ops.gelu(x, torch.empty_like(x), form)
    z = x.double()
    want = 0.5 * z * (1 + torch.erf(z / math.sqrt(2.0))) if form == "gelu" else 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))
    close(out, want, 5e-3)


@pytest.mark.parametrize("rows, dim, slices", [(1, 4, 1), (8, 2048, 3), (64, 1024, 5), (3, 8192, 2), (5, 1028, 9), (70, 2052, 0), (2, 4, 0)])
@pytest.mark.parametrize("bias, dtype", [(True, torch.float32), (False, torch.bfloat16)])
def test_layernorm_behind_a_product_left_unfinished(rows, dim, slices, bias, dtype):
    """Partial sums (more than four, fewer, one) and a bf16 product, added before the norm; without one, the same rows."""
    from runtime.kernels import ops
    x, w, b = torch.randn(rows, dim, device=DEV) + 3, torch.randn(dim, device=DEV), torch.randn(dim, device=DEV) if bias else None
    parts = torch.randn(slices, rows, dim, device=DEV) if slices else torch.randn(rows, dim, device=DEV).bfloat16()
    v = x.double() + (parts.double().sum(0) if slices else parts.double())
    out = ops.layernorm_partials(x, (parts.view(-1) if slices else parts, slices), w, torch.empty(rows, dim, device=DEV, dtype=dtype), 1e-5, bias=b)
    close(x, v, 5e-7)
    want = torch.nn.functional.layer_norm(v, (dim,), w.double(), None if b is None else b.double(), 1e-5)
    tol = 5e-6 if dtype == torch.float32 else 5e-3       # (four values of mean 3: their deviations keep 1e-6 of themselves)
    close(out, want, tol)
    close(ops.layernorm(x, w, torch.empty_like(out), 1e-5, bias=b), want, tol)


@pytest.mark.parametrize("dim", [1024, 1536, 8192])
def test_layernorm_of_a_block_a_row_is_as_close_to_64_bits_as_of_a_wave_a_row(dim):
    """The same rows 64 at a time (a block a row) and all at once (a wave a row): 2,048 rows, whose mean square errors differ by the
    forms' own roundings and by at most 1 % by chance."""
    from runtime.kernels import ops
    gen = torch.Generator(device=DEV).manual_seed(dim)
    x, w = 2 * torch.randn(2048, dim, device=DEV, generator=gen) + 1, torch.rand(dim, device=DEV, generator=gen) + 0.5
    z = x.double()
    z = z - z.mean(1, keepdim=True)
    want = z * torch.rsqrt(z.square().mean(1, keepdim=True) + 1e-5) * w.double()
    error = lambda out: ((out.double() - want).norm() / want.norm()).item()
    few = torch.cat([ops.layernorm(part, w, torch.empty_like(part), 1e-5) for part in x.split(64)])
    assert error(few) <= 1.01 * error(ops.layernorm(x, w, torch.empty_like(x), 1e-5))


@pytest.mark.parametrize("dim, heads, others", [(16, 3, 20), (32, 2, 0), (64, 5, 8), (128, 4, 260), (256, 3, 4), (128, 120, 10240), (64, 201, 13000)])
def test_short_convolution_with_unit_heads(dim, heads, others):
    """Heads whose results become unit vectors, beside channels that stay, in the kernels of few and of many inputs: against the unit vectors as a
    kernel of their own.  A step of single rows gives the same."""
    from runtime.kernels import ops
    units, taps, gates_of = dim * heads, 4, 5
    channels = units + others
    for counts, single in (([1] * 7, True), ([40, 1, 90], False)):
        T, n = sum(counts) + 2, len(counts)
        seg, starts, slots = np.concatenate([np.repeat(np.arange(n), counts), [-1] * 2]), np.concatenate(([0], np.cumsum(counts))), list(range(n))[::-1]
        wide = torch.randn(T, channels + 8, device=DEV)
        x, dt = wide[:, :channels], wide[:, channels:channels + gates_of]
        w, made = torch.randn(channels, taps, device=DEV), []
        state = torch.randn(n, (taps - 1) * channels, device=DEV)
        gate = torch.randn(gates_of, device=DEV)
        for unit in ((heads, dim, 1e-6), None):
            out, kept = torch.full((T, channels), 9.0, device=DEV), state.clone()
            step, decay = (torch.full((T, gates_of), 9.0, device=DEV) for _ in range(2))
            ops.conv_silu(x, w, None, kept, out, ints(seg), ints(starts), ints(slots), gates=(dt, gate, gate, step, decay), single_rows=single, unit=unit)
            assert (out[-2:] == 9.0).all()               # (rows of no segment stay)
            if unit is None:
                ops.unit_heads(out[:, :units], heads, dim, eps=1e-6)
            made.append((out[:-2], kept, step, decay))
        # `dim` squares are added in another order, and a root taken: a few roundings
        close(made[0][0][:, :units], made[1][0][:, :units].double(), 2e-6)
        assert torch.equal(made[0][0][:, units:], made[1][0][:, units:]) and all(torch.equal(a, b) for a, b in zip(made[0][1:], made[1][1:]))
    for bad in (8, 24, 512):
        assert not ops.conv_unit_ok(bad)
