"""An RMSNorm between two ring products, of which no kernel is made: the first product leaves its rows times the norm's weight and
their sums of squares, the second finishes the norm in its epilogue."""
import importlib

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = 2.0 ** -8          # half a unit in the last place of bf16, relative


@pytest.fixture(scope="module")
def ops():
    return importlib.import_module("runtime.kernels.ops")


def rnd(*shape, dtype=torch.float32, spread=1.0, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g, device=DEV) * spread).to(dtype)


def first(ops, m, n, k):
    """The rows that a product leaves, checked against the product followed by torch's own sums."""
    a, w = rnd(m, k, dtype=torch.bfloat16), rnd(n, k, dtype=torch.bfloat16, spread=k ** -0.5, seed=1)
    weight, x = rnd(n, seed=2) + 2.0, rnd(m, n, seed=3)
    x[m // 2] *= 1e3
    want = ops.gemm_ring(a, w, x.clone(), residual=x)
    parts = ops.lib().cisr_gemm_ring_normed_parts(m, n, k)
    assert parts in [-(-n // cols) for cols in (32, 64, 128, 256)]
    rows, sums = torch.full((m, n), 7.0, dtype=torch.bfloat16, device=DEV), torch.full((parts, m), float("nan"), device=DEV)
    ops.gemm_ring_normed(a, w, x, weight, rows, sums)
    assert torch.equal(x, want) and torch.equal(rows, (want * weight).to(torch.bfloat16))
    squares, total = want.double().square().sum(1), sums.double().sum(0)
    assert ((total - squares).abs() <= 2.0 ** -24 * 256 * squares).all()      # (at most 256 squares a sum, all positive)
    return x, weight, ops.ScaledRows(rows, sums, 1e-5)


def normed(scaled, x):
    """The rows as a 64-bit norm gives them, from the stored ones (whose rounding is the first product's)."""
    return scaled.rows.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + scaled.eps)


# rows around the tiles' edges; widths of one, of whole and of broken runs of columns; the least and a long inner size
SIZES = [(65, 64, 64), (127, 576, 576), (333, 832, 1024), (500, 932, 512), (1061, 1024, 2048), (1777, 576, 576), (2300, 960, 4096), (66, 1024, 64)]


@pytest.mark.parametrize("m, n, k", SIZES)
@pytest.mark.parametrize("inter", [64, 1536, 4100])
def test_gate_and_up_finish_the_norm(ops, m, n, k, inter):
    x, weight, scaled = first(ops, m, n, k)
    if n % 64:          # (no inner size of the ring product)
        return
    w = rnd(2 * inter, n, dtype=torch.bfloat16, spread=n ** -0.5, seed=4)
    at = ops._ring_operands(scaled.rows, w, out := torch.empty(m, inter, dtype=torch.bfloat16, device=DEV))
    ops._ring_gated(at, m, inter, n, out, None, sums=scaled.args(m))
    product = (normed(scaled, x) @ w.double().t())
    gate, up = product[:, :inter], product[:, inter:]
    want = gate * torch.sigmoid(gate) * up
    # gate and up are rounded to bf16 (and their float sums may round the other way: twice that), so is the result
    tol = 3 * BF * ((gate.abs() + 1) * up.abs() * 1.1 + gate.abs() * up.abs()) + 2.0 ** -20 * n ** 0.5 + BF * want.abs()
    assert ((out.double() - want).abs() <= tol).all()
    if ops.ring_gated_ok(scaled.rows, w):
        assert torch.equal(ops.gemm_swiglu(scaled, w, torch.empty_like(out)), out)


@pytest.mark.parametrize("m, n, k", [s for s in SIZES if s[1] % 64 == 0 and s[0] > 65])
@pytest.mark.parametrize("heads, kv, dim", [(9, 3, 64), (8, 2, 128)])
def test_projection_and_rotation_finish_the_norm(ops, m, n, k, heads, kv, dim):
    x, weight, scaled = first(ops, m, n, k)
    w = rnd((heads + 2 * kv) * dim, n, dtype=torch.bfloat16, spread=n ** -0.5, seed=5)
    page, pages = 16, -(-m // 16)
    positions = torch.arange(m, dtype=torch.int32, device=DEV)
    angle = torch.arange(m, device=DEV)[:, None] * 10000.0 ** (-torch.arange(0, dim, 2, device=DEV) / dim)
    cos, sin = angle.cos().float().contiguous(), angle.sin().float().contiguous()
    kc, vc = (torch.zeros(pages, kv, *s, dtype=torch.bfloat16, device=DEV) for s in ((page, dim), (dim, page)))
    q = torch.empty(m, heads * dim, dtype=torch.bfloat16, device=DEV)
    ops.qkv_rope(scaled, w, q, positions, positions, cos, sin, kc, vc, heads, kv, dim, page)
    product = (normed(scaled, x) @ w.double().t()).view(m, heads + 2 * kv, dim)
    a, b = product[..., :dim // 2], product[..., dim // 2:]
    c, s = cos.double()[:, None], sin.double()[:, None]
    turned = torch.cat([a * c - b * s, b * c + a * s], -1)
    def near(got, want):
        assert ((got.double() - want).abs() <= BF * want.abs() + 2.0 ** -18).all()
    near(q.view(m, heads, dim), turned[:, :heads])
    near(kc.permute(0, 2, 1, 3).reshape(-1, kv, dim)[:m], turned[:, heads:heads + kv])
    near(vc.permute(0, 3, 1, 2).reshape(-1, kv, dim)[:m], product[:, heads + kv:])


def test_what_is_refused(ops):
    x, weight, scaled = first(ops, 129, 576, 576)
    a, w = rnd(129, 576, dtype=torch.bfloat16), rnd(576, 576, dtype=torch.bfloat16)
    out = torch.empty(129, 288, dtype=torch.bfloat16, device=DEV)
    for rows, sums in ((scaled.rows[:64], scaled.sums[:, :64].contiguous()), (scaled.rows, scaled.sums[:-1]), (scaled.rows[:, :-4], scaled.sums)):
        with pytest.raises(ops.KernelError):
            ops.gemm_ring_normed(a, w, x, weight, rows, sums)
    with pytest.raises(ops.KernelError):        # too few rows for the ring product
        ops.gemm_swiglu(ops.ScaledRows(scaled.rows[:16], scaled.sums[:, :16].contiguous(), 1e-5), w, out[:16])
    assert ops.ring_normed_parts(a[:64], w, x[:64], weight) == 0
    assert ops.ring_normed_parts(a, w, x, torch.cat([weight, weight])[1:577]) == 0
