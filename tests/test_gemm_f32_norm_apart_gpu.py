"""Where the norm of 32-bit rows is a kernel of its own again (many results), the parts run it so; the products still take what they took."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_parts_run_the_norm_apart_where_that_is_faster_and_the_products_still_take_it():
    from runtime.kernels import ops
    from runtime.parts import GatedMLP, LMHead, RMSNorm
    rows, K, N = 1024, 64, 2048
    g = torch.Generator(device=DEV).manual_seed(0)
    x = torch.randn(rows, K, device=DEV, generator=g)
    norm = RMSNorm("n", K, 1e-5)
    norm.weight = 1.0 + 0.1 * torch.randn(K, device=DEV, generator=g)
    w = torch.randn(N, K, device=DEV, generator=g) * K ** -0.5
    ffn, head = GatedMLP("f", K, N // 2), LMHead("h", N, K)
    ffn.w_gate_up = head.weight = w
    index = torch.arange(rows, dtype=torch.int32, device=DEV)
    for count, fused in ((512, True), (rows, False)):
        assert ffn.fuses_norm(norm, x[:count], None) is fused and head.fuses_norm(norm, x, index[:count]) is fused
    want = x.double() * torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-5) * norm.weight.double() @ w.double().T
    off = lambda got, want: ((got.double() - want).norm() / want.norm()).item()
    # sums of K products in at least eight runs, an operand and a result rounded once more: 3e-7 (as test_gemm_f32_norm_gpu)
    assert off(ops.gemm_normed(x, (norm.weight, 1e-5, index), w, torch.empty(rows, N, device=DEV)), want) < 1e-6
    gated = ops.gemm_swiglu(x, w, torch.empty(rows, N // 2, device=DEV), norm=(norm.weight, 1e-5, None))
    assert off(gated, torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:]) < 1e-6
