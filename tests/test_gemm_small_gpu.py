"""gemm_small.hip against an fp64 product: every tile at its edges."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops.kernels import small_tile

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (M, N, K): each tile of the rule (2 to 5: the ring, at one row and few, many and long K-steps; its own tiles:
# test_ring_tiles_gpu.py) at one row, ragged rows and columns, the shortest K, few and many K-steps
SHAPES = {0: [(1, 4, 512), (1, 768, 768), (17, 772, 576), (64, 768, 3072), (16, 36, 448)],
          1: [(19, 2304, 768), (33, 2036, 512), (128, 768, 1088), (40, 2020, 704)],
          2: [(1, 4, 64), (130, 2308, 192), (320, 1024, 64), (320, 1792, 768)], 3: [(300, 3076, 64), (870, 768, 1024), (2048, 2304, 768)],
          4: [(1025, 1028, 1088), (1500, 768, 3072)], 5: [(2500, 1028, 1088), (4096, 768, 3072)],
          6: [(256, 768, 3072), (33, 3076, 384), (65, 2304, 768), (129, 1028, 448)],
          7: [(257, 1028, 1088), (512, 768, 3072), (129, 2308, 384)], 8: [(870, 768, 3072), (513, 1028, 1152), (1024, 1024, 4096)]}


@pytest.mark.parametrize("tile,M,N,K", [(t, *s) for t, v in SHAPES.items() for s in v])
@pytest.mark.parametrize("gelu,bias,res", [(False, True, True), (True, True, False), (False, False, False)])
def test_gemm_small(tile, M, N, K, gelu, bias, res):
    assert small_tile(M, N, K) == (ops.native().RING_TILE if 2 <= tile <= 5 else tile)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)

    def rnd(*shape, pad=0, scale=1.0):  # a view of wider rows: strides other than the width
        t = torch.randn(*shape[:-1], shape[-1] + pad, device=DEV, generator=g) * scale
        return t.to(torch.bfloat16)[..., :shape[-1]]

    A, B = rnd(M, K, pad=8), rnd(N, K, pad=16, scale=K ** -0.5)
    b = rnd(N) if bias else None
    r = rnd(M, N, pad=4) if res else None
    out = rnd(M, N, pad=12)
    guard = out.clone()
    wide = torch.empty(M + 1, N + 12, dtype=torch.bfloat16, device=DEV).fill_(7.0)
    dst = wide[:M, :N]
    ops.gemm_bt(A, B, bias=b, residual=r, epilogue=ops.EPI_GELU if gelu else ops.EPI_NONE, out=dst)
    exp = A.double() @ B.double().t()
    if bias:
        exp = exp + b.double()
    if gelu:
        exp = torch.nn.functional.gelu(exp)
    # two roundings to bf16 (2^-8 of the value each: the product's and, with a residual, the sum's) and fp32 sums of
    # K products of size about K^-1/2 (error far below 1e-4 at these K)
    tol = 2.0 ** -8 * exp.abs() + 1e-4
    if res:
        exp = exp + r.double()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((dst.double() - exp).abs() <= tol).all()
    assert (wide[M:] == 7.0).all() and (wide[:, N:] == 7.0).all() and torch.equal(out, guard)
    assert torch.equal(ops.gemm_bt(A, B, bias=b, residual=r, epilogue=ops.EPI_GELU if gelu else ops.EPI_NONE), dst)
