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
