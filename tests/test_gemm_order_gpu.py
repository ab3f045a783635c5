"""Projections whose input is larger than half the Infinity Cache walk their tiles in blocks of columns: the same bits."""
import pytest
import torch

from django_assistant_bot_amd import ops

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
