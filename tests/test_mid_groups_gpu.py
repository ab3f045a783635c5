"""gemm_mid on fewer groups than fit the chip."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one to eight row tiles; equal parts of a tile, whole tiles, fewer groups than tiles, parts of unequal length
@pytest.mark.parametrize("M,N,K", [(1, 2048, 2048), (130, 2048, 2048), (257, 3072, 2048), (300, 512, 4096), (384, 4096, 4096),
                                   (777, 768, 3072), (1000, 3072, 2048), (500, 6144, 1024)])
@pytest.mark.parametrize("glu", [False, True])
def test_fewer_groups(M, N, K, glu):
    tm = -(-M // 128)
    assert 0 < ops.kernels.native().gemm_mid_groups(M, N, K) < 8 * (32 // tm)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    A = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    W = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    B = ops.shuffle_weights(W, 8 if glu else 1)
    res = None if glu else torch.randn(M, N, device=DEV, generator=g).to(torch.bfloat16)
    exp = A.float() @ W.float().t()
    # bf16 rounding of the product (2^-8) and of the sum or the activation; fp32 sums far below
    if glu:
        v = exp.view(M, N // 16, 2, 8)
        exp = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
        tol = 2.0 ** -8 * exp.abs() + 1e-4
    else:
        tol = 2.0 ** -8 * exp.abs() + 1e-4
        exp = exp + res.float()
        tol = tol + 2.0 ** -8 * exp.abs()
    first = None
    for _ in range(3):  # the ready flags are down again after each launch
        out = ops.kernels.gemm_mid(A, B, residual=res, epilogue=ops.EPI_SWIGLU8 if glu else ops.EPI_NONE, b_group=8 if glu else 1)
        assert ((out.float() - exp).abs() <= tol).all()
        first = out if first is None else first
        assert torch.equal(out, first)
