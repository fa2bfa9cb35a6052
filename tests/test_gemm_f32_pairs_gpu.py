"""The 32-bit products with two rows of W a column, the activation or the rotation as their epilogue, against the product and the kernel
behind it (the same sums, in the same order) and against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def off(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("rows, inter, K", [(1, 16, 4), (2, 1536, 576), (17, 33, 70), (130, 1536, 576), (130, 40, 1100), (700, 1030, 260)])
def test_gated_product(rows, inter, K):
    from runtime.kernels import ops
    a, w = torch.randn(rows, K, device=DEV), torch.randn(2 * inter, K, device=DEV) * K ** -0.5
    out = torch.full((rows, inter), float("nan"), device=DEV)
    both = torch.empty(rows, 2 * inter, device=DEV)
    ops.gemm_swiglu(a, w, out, gate_up=both)
    apart = torch.empty_like(out)
    ops.swiglu(ops.gemm(a, w, torch.empty_like(both)), apart)
    z = a.double() @ w.double().T
    want = torch.nn.functional.silu(z[:, :inter]) * z[:, inter:]
    # sums of K products in at least eight runs: 3e-7; the exponential's and the quotient's roundings are of that size
    assert off(out, want) < 1e-6 and off(out, want) < 1.05 * off(apart, want) + 1e-9
    assert torch.equal(out, apart)
    with pytest.raises(ops.KernelError):
        ops.gemm_swiglu(a, w, out)


@pytest.mark.parametrize("rows, heads, kv_heads, dim, K, own", [(1, 9, 3, 64, 576, True), (3, 2, 1, 40, 44, True), (130, 9, 3, 64, 576, True),
                                                                (33, 4, 4, 32, 1028, False), (300, 8, 2, 128, 512, True)])
def test_projection_with_rotation_and_pages(rows, heads, kv_heads, dim, K, own):
    from runtime.kernels import ops
    page, pages = 8, -(-rows // 8) + 2
    g = torch.Generator(device=DEV).manual_seed(rows)
    n_kv = kv_heads if own else 0
    a = torch.randn(rows, K, device=DEV, generator=g)
    w = torch.randn((heads + 2 * n_kv) * dim, K, device=DEV, generator=g) * K ** -0.5
    pos = torch.randint(0, 500, (rows,), device=DEV, generator=g, dtype=torch.int32)
    slots = torch.randperm(pages * page, device=DEV, generator=g)[:rows].int()
    slots[rows // 2] = -1
    angle = torch.arange(500, device=DEV, dtype=torch.float64)[:, None] * 10000.0 ** (-torch.arange(dim // 2, device=DEV, dtype=torch.float64) * 2 / dim)
    cos, sin = angle.cos().float(), angle.sin().float()
    made = []
    for fused in (True, False):
        k, v = torch.full((pages, kv_heads, page, dim), 7.0, device=DEV), torch.full((pages, kv_heads, dim, page), 7.0, device=DEV)
        cache = (k, v) if own else (None, None)
        if fused:
            q = torch.full((rows, heads * dim), float("nan"), device=DEV)
            assert ops.qkv_rope_f32_ok(a, w, dim, cos)
            ops.qkv_rope(a, w, q, pos, slots if own else None, cos, sin, *cache, heads, kv_heads, dim, page)
        else:
            both = ops.gemm(a, w, torch.empty(rows, w.shape[0], device=DEV))
            ops.rope_scatter(both, pos, slots if own else None, cos, sin, *cache, heads, kv_heads, dim, page)
            q = both[:, :heads * dim].contiguous()
        made.append((q, k, v))
    # the same sums, and the rotation's two products and sum are contracted alike
    for x, y in zip(*made):
        assert torch.isfinite(x).all() and torch.equal(x, y)
    z = (a.double() @ w.double().T)[:, :heads * dim].view(rows, heads, dim)
    c, s = cos.double()[pos.long()][:, None], sin.double()[pos.long()][:, None]
    lo, hi = z[..., :dim // 2], z[..., dim // 2:]
    assert off(made[0][0].view(rows, heads, dim), torch.cat([lo * c - hi * s, hi * c + lo * s], -1)) < 1e-6


def test_gated_product_refuses_and_takes_what_it_did_with_two_kernels():
    """The buffer for the product of gate and up is checked although nothing is written to it; a result may lie where the rows were."""
    from runtime.kernels import ops
    rows, width = 19, 48
    a, w = torch.randn(rows, width, device=DEV), torch.randn(2 * width, width, device=DEV)
    both, out = torch.empty(rows, 2 * width, device=DEV), torch.empty(rows, width, device=DEV)
    for wrong in (both[:, :width], both[:-1], both.double(), both.bfloat16(), both.cpu(), torch.empty(2 * width, rows, device=DEV).t()):
        with pytest.raises(ops.KernelError):
            ops.gemm_swiglu(a, w, out, gate_up=wrong)
    ops.gemm_swiglu(a, w, out, gate_up=both)
    ops.gemm_swiglu(a, w, a, gate_up=both)
    assert torch.equal(a, out)
