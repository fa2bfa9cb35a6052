"""The 32-bit products with the RMSNorm of their rows fused, against 64 bits and the norm as a kernel of its own."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def off(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


def normed(x, weight, eps):
    return x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + eps) * weight.double()


# tiles of 1 x 1 to 4 x 4 and beyond one round, inner sizes that end inside a sixteen, the largest
@pytest.mark.parametrize("rows, cols, K", [(1, 16, 4), (2, 3072, 576), (16, 960, 576), (17, 576, 580), (130, 3072, 576), (192, 3072, 576), (256, 3072, 576),
                                           (333, 960, 576), (512, 3072, 576), (2, 2048, 1020), (500, 960, 1020), (300, 2500, 540), (130, 6144, 132)])
def test_norm_inside_the_product(rows, cols, K):
    from runtime.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    wide = torch.randn(rows + 5, K + 8, device=DEV, generator=g) * 3.0
    x = wide[:, :K]                                   # (rows of a wider matrix)
    weight = 1.0 + 0.1 * torch.randn(K, device=DEV, generator=g)
    w = torch.randn(cols, K, device=DEV, generator=g) * K ** -0.5
    index = torch.randperm(rows + 5, device=DEV, generator=g)[:rows].int()
    assert ops.fused_norm_ok(x, w, rows, weight)
    out = ops.gemm_normed(x, (weight, 1e-5, index), w, torch.full((rows, cols), float("nan"), device=DEV))
    want = normed(x[index.long()], weight, 1e-5) @ w.double().T
    h = ops.rmsnorm(x.contiguous(), weight, torch.empty(rows, K, device=DEV), 1e-5, index)
    apart = ops.gemm(h, w, torch.empty(rows, cols, device=DEV))
    # sums of K products in at least eight runs: 3e-7 (test_gemm_f32_pairs_gpu); the norm rounds an operand once and a result once where the
    # kernel of its own rounds an operand twice, so it is no further off but for chance (few outputs: 5 in 100 more)
    assert off(out, want) < 1e-6 and off(out, want) < 1.05 * off(apart, want) + 2e-8
    some = sorted({0, max(rows - 16, 0), rows // 32 * 16})
    for at in some:                                   # a row's bits are its own, whatever the tile
        assert torch.equal(out[at:at + 16], ops.gemm_normed(x, (weight, 1e-5, index[at:at + 16].clone()), w, torch.empty_like(out[at:at + 16])))
    if cols % 2 == 0:
        x = x[:rows]
        gated = ops.gemm_swiglu(x, w, torch.full((rows, cols // 2), float("nan"), device=DEV), norm=(weight, 1e-5, None))
        z = normed(x, weight, 1e-5) @ w.double().T
        assert off(gated, torch.nn.functional.silu(z[:, :cols // 2]) * z[:, cols // 2:]) < 1e-6


@pytest.mark.parametrize("rows, heads, kv, dim, K", [(1, 9, 3, 64, 576), (130, 9, 3, 64, 576), (333, 9, 3, 64, 576), (70, 8, 2, 128, 1008)])
def test_norm_inside_the_projection(rows, heads, kv, dim, K):
    """Queries, keys and values with the norm fused are those of the product's own rows, bit for bit where only the norm differs by rounding: 1e-6."""
    from runtime.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(rows)
    x, weight = torch.randn(rows, K, device=DEV, generator=g), 1.0 + 0.1 * torch.randn(K, device=DEV, generator=g)
    w = torch.randn((heads + 2 * kv) * dim, K, device=DEV, generator=g) * K ** -0.5
    pos = torch.randint(0, 200, (rows,), device=DEV, generator=g, dtype=torch.int32)
    pages = -(-rows // 16) + 1
    slots = torch.randperm(pages * 16, device=DEV, generator=g)[:rows].int()
    angle = torch.rand(200, dim // 2, device=DEV, generator=g) * 6.3
    cos, sin = angle.cos(), angle.sin()
    made = []
    for fused in (True, False):
        k, v = torch.full((pages, kv, 16, dim), 7.0, device=DEV), torch.full((pages, kv, dim, 16), 7.0, device=DEV)
        q = torch.full((rows, heads * dim), float("nan"), device=DEV)
        a = x if fused else ops.rmsnorm(x, weight, torch.empty_like(x), 1e-5)
        assert ops.qkv_rope_fused_ok(a, w, dim, cos, fused, weight=weight) or not fused
        ops.qkv_rope(a, w, q, pos, slots, cos, sin, k, v, heads, kv, dim, 16, norm=(weight, 1e-5) if fused else None)
        made.append((q, k, v))
    for one, other in zip(*made):
        assert torch.isfinite(one).all() and off(one, other.double()) < 1e-6


def test_what_the_fused_norm_takes():
    from runtime.kernels import ops
    x, w, weight = torch.randn(4, 64, device=DEV), torch.randn(32, 64, device=DEV), torch.ones(65, device=DEV)
    out = torch.empty(4, 32, device=DEV)
    assert ops.fused_norm_ok(x, w, 4, weight[:64]) and not ops.fused_norm_ok(x, w, 4, weight[1:])
    assert not ops.fused_norm_ok(torch.randn(4, 1024, device=DEV), torch.randn(32, 1024, device=DEV), 4)      # (sixteen waves a tile)
    assert not ops.fused_norm_ok(x[:, :62], w[:, :62], 4) and not ops.fused_norm_ok(torch.randn(4, 65, device=DEV)[:, :64], w, 4)
    for bad in ((weight[1:], 1e-5, None), (weight[:63], 1e-5, None)):
        with pytest.raises(ops.KernelError):
            ops.gemm_normed(x, bad, w, out)
    with pytest.raises(ops.KernelError):
        ops.gemm_normed(x, (weight[:64], 1e-5, None), w, out.bfloat16())
    # a row of zeros and one that is not finite are their own affair
    x[1] = 0.0
    x[2, 5] = float("nan")
    got = ops.gemm_normed(x, (weight[:64], 1e-5, None), w, out)
    assert (got[1] == 0).all() and torch.isnan(got[2]).all() and torch.isfinite(got[[0, 3]]).all()
