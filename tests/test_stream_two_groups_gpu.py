"""The 64-row tiles of the decode GEMM with two k-groups (33-64 and 65-128 rows) against an fp32 product."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
ROWS = [(12, 33), (12, 48), (12, 64), (9, 65), (9, 100), (9, 128)]


def _operands(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    return x, w, x.float() @ w.float().t(), torch.randn(N, device=DEV, generator=g)


@pytest.mark.parametrize("cfg,M", ROWS)
@pytest.mark.parametrize("N,K", [(256, 256), (16384, 2048), (384, 1152)])
@pytest.mark.parametrize("bias", [False, True])
def test_gated_on_the_grouped_copy(cfg, M, N, K, bias):
    x, w, exp, gb = _operands(M, N, K)
    v = exp.view(M, N // 16, 2, 8)
    if bias:
        v = v + gb.view(2, N // 16, 8).transpose(0, 1)
    exp = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
    out = torch.full((M + 1, N // 2), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.stream_gemm(x, ops.shuffle_weights(w, 8), epilogue=ops.EPI_SWIGLU8, nt=True, cfg=cfg, w_group=8, out=out[:M],
                    glu_bias=gb if bias else None)
    # one rounding to bf16 (2^-8 of the value); the fp32 sums and the gate are far below 1e-4
    assert ((out[:M].float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4).all() and (out[M] == 7.0).all()


@pytest.mark.parametrize("cfg,M", ROWS[:3])
@pytest.mark.parametrize("N,K,S", [(64, 128, 1), (192, 1024, 4), (4096, 4096, 4), (2048, 2048, 8), (1024, 8192, 16)])
def test_slices(cfg, M, N, K, S):
    x, w, exp, _ = _operands(M, N, K)
    y = ops.stream_gemm(x, ops.shuffle_weights(w), splits=S, nt=True, cfg=cfg, **({"slab_dtype": torch.bfloat16} if S > 1 else {}))
    # a bf16 rounding (2^-8) of the result, or of each of the S partial sums
    got = y.float().sum(0) if S > 1 else y.float()
    tol = 2.0 ** -8 * (y.float().abs().sum(0) if S > 1 else exp.abs()) + 1e-4
    assert got.shape == exp.shape and ((got - exp).abs() <= tol).all()
