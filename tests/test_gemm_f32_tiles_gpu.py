"""The tiles of the 32-bit products: whatever tile the rule picks, a row has the bits that it has in a step of sixteen rows, and the
sums are those of 64 bits but for their roundings."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# rows and sizes at either side of the rule's lines: 1 x 1, 1 x 2, 2 x 2, 3 x 2, 4 x 2, beyond one round; sixteen waves; not aligned
@pytest.mark.parametrize("rows, N, K", [(17, 576, 576), (113, 576, 576), (128, 576, 576), (192, 576, 576), (289, 576, 576), (500, 576, 576),
                                        (512, 960, 576), (700, 960, 576), (64, 576, 1536), (192, 576, 1536), (320, 576, 1536), (512, 576, 1536),
                                        (64, 2048, 1024), (192, 2048, 1024), (300, 2500, 1040), (200, 4200, 1024), (130, 900, 75), (700, 1000, 1030)])
def test_bits_of_a_row_do_not_depend_on_the_tile(rows, N, K):
    from runtime.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(rows + N)
    a, w = torch.randn(rows, K, device=DEV, generator=g), torch.randn(N, K, device=DEV, generator=g)
    r = torch.randn(rows, N, device=DEV, generator=g)
    out = ops.gemm(a, w, r.clone(), residual=r)
    # at most K roundings of half an ulp of a sum below 8 sqrt(K)
    assert (out.double() - r.double() - a.double() @ w.double().T).abs().max().item() <= K * 2.0 ** -24 * 8 * K ** 0.5
    some = [0, rows // 2 // 16 * 16, rows - 16]
    for at in some:
        assert torch.equal(out[at:at + 16], ops.gemm(a[at:at + 16], w, torch.empty(16, N, device=DEV), residual=r[at:at + 16]))
    if N % 2 == 0:
        gated = ops.gemm_swiglu(a, w, torch.empty(rows, N // 2, device=DEV), gate_up=torch.empty(rows, N, device=DEV))
        for at in some:
            assert torch.equal(gated[at:at + 16], ops.gemm_swiglu(a[at:at + 16], w, torch.empty(16, N // 2, device=DEV), gate_up=torch.empty(16, N, device=DEV)))


# (cols = both rows of W of a pair: gated 3,072 x 576, 1,536 x 1,040; 9 + 2 x 3 heads of 64, 8 + 2 x 2 heads of 128) rows and the tile they take
@pytest.mark.parametrize("rows, inter, K", [(20, 1536, 576), (60, 1536, 576), (100, 1536, 576), (200, 1536, 576), (300, 1536, 576), (400, 1536, 576), (1100, 1536, 576),
                                            (40, 768, 1040), (150, 768, 1040), (310, 768, 1040), (400, 768, 1040), (560, 768, 1040), (520, 1536, 577), (70, 1536, 577)])
def test_bits_of_a_gated_row_do_not_depend_on_the_tile(rows, inter, K):
    """1 x 2, 2 x 2, 4 x 2, 3 x 4, 4 x 4, beyond one round 2 x 2 and 2 x 4; sixteen waves; not aligned.  A row alone among sixteen has the same."""
    from runtime.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    a, w = torch.randn(rows, K, device=DEV, generator=g), torch.randn(2 * inter, K, device=DEV, generator=g) * K ** -0.5
    gu = torch.empty(rows, 2 * inter, device=DEV)
    out = ops.gemm_swiglu(a, w, torch.full((rows + 1, inter), 7.0, device=DEV)[:rows], gate_up=gu)
    for at in sorted({0, rows // 2 // 16 * 16, rows - 16}):
        assert torch.equal(out[at:at + 16], ops.gemm_swiglu(a[at:at + 16], w, torch.empty(16, inter, device=DEV), gate_up=gu[:16]))
    gate, up = (a.double() @ x.double().T for x in (w[:inter], w[inter:]))
    want = torch.nn.functional.silu(gate) * up
    # gate and up: at most K roundings of half an ulp of sums below 8; the activation's slope is below 1.1, and it rounds three times
    bound = K * 2.0 ** -24 * 8 * (1.1 * up.abs() + gate.abs()) + 2.0 ** -21 * want.abs() + 1e-6
    assert ((out.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("rows, K, heads, kv, dim", [(17, 576, 9, 3, 64), (100, 576, 9, 3, 64), (192, 576, 9, 3, 64), (300, 576, 9, 3, 64), (400, 576, 9, 3, 64), (560, 576, 9, 3, 64),
                                                     (1000, 576, 9, 3, 64), (1200, 576, 9, 3, 64), (3300, 576, 9, 3, 64), (60, 1040, 8, 2, 128), (200, 1040, 8, 2, 128),
                                                     (310, 1040, 8, 2, 128), (400, 1040, 8, 2, 128), (560, 1040, 8, 2, 128), (1100, 577, 9, 3, 64), (130, 577, 9, 3, 64)])
def test_bits_of_a_turned_row_do_not_depend_on_the_tile(rows, K, heads, kv, dim):
    """1 x 1, 1 x 2, 2 x 2, 3 x 2, 4 x 2, 3 x 4, 4 x 4, 2 x 2 and 2 x 4 beyond one round; sixteen waves; not aligned: queries, key and value pages
    of all rows at once and of sixteen at a time."""
    from runtime.kernels import ops
    g = torch.Generator(device=DEV).manual_seed(rows + K)
    a, w = torch.randn(rows, K, device=DEV, generator=g), torch.randn((heads + 2 * kv) * dim, K, device=DEV, generator=g)
    angle = torch.rand(rows + 3, dim // 2, device=DEV, generator=g) * 6.3
    cos, sin = angle.cos(), angle.sin()
    positions = torch.randperm(rows + 3, device=DEV, generator=g)[:rows].int()
    page = 16
    slots = torch.arange(rows, device=DEV, dtype=torch.int32)

    def run(parts):
        q = torch.empty(rows, heads * dim, device=DEV)
        keys, values = torch.zeros(rows // page + 1, kv, page, dim, device=DEV), torch.zeros(rows // page + 1, kv, dim, page, device=DEV)
        for lo, hi in parts:
            ops.qkv_rope(a[lo:hi], w, q[lo:hi], positions[lo:hi].contiguous(), slots[lo:hi].contiguous(), cos, sin, keys, values, heads, kv, dim, page)
        return q, keys, values
    whole = run([(0, rows)])
    for got, want in zip(run([(at, min(at + 16, rows)) for at in range(0, rows, 16)]), whole):
        assert torch.equal(got, want)
    x, y = (a.double() @ w.double().T)[:, :heads * dim].view(rows, heads, 2, dim // 2).unbind(2)
    c, s = (t.double()[positions.long()][:, None] for t in (cos, sin))
    turned = torch.stack((x * c - y * s, y * c + x * s), 2).view(rows, -1)
    assert (whole[0].double() - turned).abs().max().item() <= 2 * K * 2.0 ** -24 * 8 * K ** 0.5
