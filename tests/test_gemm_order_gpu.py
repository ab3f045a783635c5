"""The tile orders of the 256 x 256 GEMM (blocks of columns for an input larger than half the Infinity Cache, even groups of rows
for many columns): every tile once, the same bits."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops.kernels import gemm256

pytestmark = pytest.mark.gpu
DEV = "cuda"


# 1 to 5 tile columns (blocks of 3 and what is left over), tile rows that are and are not whole groups of 8, a ragged last tile
@pytest.mark.parametrize("M,N", [(524288, 256), (524288 + 2048, 768), (524288 + 77, 1024), (526591, 1280)])
def test_every_tile_once(M, N):
    K = 128
    g = torch.Generator(device=DEV).manual_seed(N)
    a = torch.empty(M, K, device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    w = torch.empty(N, K, device=DEV, dtype=torch.bfloat16).normal_(0, K ** -0.5, generator=g)
    b = torch.randn(N, device=DEV, generator=g).to(torch.bfloat16)
    out = torch.full((M + 1, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_bt(a, w, bias=b, out=out[:M])
    assert torch.isnan(out[M]).all()
    half = 262144  # whole tiles; each part is below the bound, in the order of rows
    for rows in (slice(0, half), slice(half, M)):
        assert a[rows].numel() * 2 < 1 << 27
        assert torch.equal(out[rows], ops.gemm_bt(a[rows], w, bias=b))
    at = torch.cat([torch.arange(512), torch.arange(M - 512, M)]).to(DEV)
    exp = a[at].double() @ w.double().t() + b.double()
    slack = K * 2.0 ** -23 * (a[at].double().abs() @ w.double().abs().t() + b.double().abs())
    assert ((out[at].double() - exp).abs() <= 2.0 ** -8 * exp.abs() + slack).all()


# one group of 1 and of 6 tile rows, 4 + 4, 5 + 5, 5 + 5 + 3; more than 256 workgroups and fewer
@pytest.mark.parametrize("M", [1, 1281, 1793, 2305, 3100])
@pytest.mark.parametrize("cols", [64, 67])
def test_even_groups_of_rows(M, cols):
    K, N = 128, 256 * cols
    g = torch.Generator(device=DEV).manual_seed(M + cols)
    a = torch.empty(M, K, device=DEV, dtype=torch.bfloat16).normal_(generator=g)
    w = ops.shuffle_weights(torch.empty(N, K, device=DEV, dtype=torch.bfloat16).normal_(0, K ** -0.5, generator=g))
    for epi in (ops.EPI_NONE, ops.EPI_SWIGLU8):
        out = gemm256(a, w, epilogue=epi, shuffled=True)
        at = N // 512 * 256  # (halves of the weights' rows: groups of 4 tile rows)
        parts = [gemm256(a, x, epilogue=epi, shuffled=True) for x in (w[:at], w[at:])]
        assert torch.isfinite(out.float()).all() and torch.equal(out, torch.cat(parts, 1))
