"""The factor of a row in an RMSNorm that a product finishes, in every kernel that has it, against 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# float products; narrow and skinny products of bf16 weights, the matrix-vector kernel (8 MB)
@pytest.mark.parametrize("dtype, K, rows", [(torch.float32, 64, 3), (torch.float32, 576, 40), (torch.bfloat16, 64, 3), (torch.bfloat16, 576, 1),
                                            (torch.bfloat16, 576, 40), (torch.bfloat16, 2048, 2), (torch.bfloat16, 2048, 12)])
@pytest.mark.parametrize("power", [-66, -40, 0, 50])
def test_factor_of_rows_of_any_size(dtype, K, rows, power):
    """Rows of c and -c and no eps: the squares and their sums are exact, so results are c times the factor, that is 1 and -1.  The mean rounds
    twice, the root is within one unit, its step and the product round once each: 3 units in the last place; means below the
    normal numbers have 17 bits (2 ** -132)."""
    from runtime.kernels import ops
    c = 2.0 ** power * (1.0 + torch.arange(rows, device=DEV) % 16 / 16.0)
    sign = (torch.arange(K, device=DEV) % 2 * 2.0 - 1.0)
    x = c[:, None] * sign
    w = torch.eye(K, device=DEV, dtype=dtype)
    weight = torch.ones(K, device=DEV)
    assert ops.fused_norm_ok(x, w, rows, weight)
    out = ops.gemm_normed(x, (weight, 0.0, None), w, torch.full((rows, K), float("nan"), device=DEV))
    assert (out - sign).abs().max() <= (2.0 ** -17 if power == -66 else 3 * 2.0 ** -23)
