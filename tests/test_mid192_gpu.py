"""gemm_mid's kernel with tiles of 192 rows (variant 192) against an fp32 product."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"
# one row; a first half of the tile alone, ragged, whole; whole tiles a group, parts of equal length, parts of unequal length and
# more behind them; an odd number of pairs of K-steps; the most row tiles
SHAPES = [(1, 2048, 1024), (128, 2048, 8192), (192, 4096, 1024), (193, 6144, 3072), (1300, 10240, 1152), (700, 28672, 1024),
          (1093, 4096, 14336), (1430, 6144, 4096), (4096, 2048, 2048)]


def _case(M, N, K, group):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    A = torch.randn(M, K + 8, device=DEV, generator=g).to(torch.bfloat16)[:, :K]  # rows with a stride of their own
    W = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    return A, ops.shuffle_weights(W, group), A.float() @ W.float().t()


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("group", [1, 8])
def test_against_the_product(M, N, K, group):
    A, B, exp = _case(M, N, K, group)
    res = torch.randn(M, N, device=DEV).to(torch.bfloat16)
    wide = torch.full((M + 1, N + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    first = None
    for _ in range(3):  # the ready flags are down again after each launch, and the order of the sums is fixed
        kernels.gemm_mid(A, B, variant=192, b_group=group, out=wide[:M, :N])
        # one rounding to bf16 (2^-8 of the value); the fp32 sums are far below 1e-4
        assert ((wide[:M, :N].float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4).all()
        first = wide[:M, :N].clone() if first is None else first
        assert torch.equal(wide[:M, :N], first)
    assert (wide[M:] == 7.0).all() and (wide[:, N:] == 7.0).all()
    out = kernels.gemm_mid(A, B, residual=res, variant=192, b_group=group)
    assert torch.equal(out, (first.float() + res.float()).to(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("epilogue", kernels.GLU8)
@pytest.mark.parametrize("bias", [False, True])
def test_glu(M, N, K, epilogue, bias):
    A, B, exp = _case(M, N, K, 8)
    v = exp.view(M, N // 16, 2, 8)
    gate, up = v[:, :, 0].reshape(M, N // 2), v[:, :, 1].reshape(M, N // 2)
    b = torch.randn(N, device=DEV) if bias else None
    if bias:
        gate, up = gate + b[:N // 2], up + b[N // 2:]
    act = {ops.EPI_SWIGLU8: torch.nn.functional.silu, ops.EPI_REGLU8: torch.relu}.get(
        epilogue, lambda t: torch.nn.functional.gelu(t, approximate="tanh"))
    exp = act(gate) * up
    out = kernels.gemm_mid(A, B, epilogue=epilogue, variant=192, b_group=8, glu_bias=b)
    # one rounding to bf16; the sums' 1e-4 of either factor times the other's size, at most 8 or so
    assert ((out.float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-3).all()


@pytest.mark.parametrize("variants", [(192, 256), (192, 64), (192, 192)])
def test_kernels_in_turn(variants):
    """The three kernels share a workspace: flags, counts and partial tiles of one mean nothing to the next."""
    A, B, exp = _case(1093, 4096, 14336, 1)
    for _ in range(4):
        for variant in variants:
            out = kernels.gemm_mid(A, B, variant=variant)
            assert ((out.float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4).all()


def test_sizes_that_the_tiles_do_not_take():
    """Column tiles that the XCDs cannot share evenly, and rows 2^23 elements apart, are the 128-row kernel's."""
    A, B, exp = _case(700, 2304, 1024, 1)
    assert torch.equal(kernels.gemm_mid(A, B, variant=192), kernels.gemm_mid(A, B, variant=64))
    A, B, _ = _case(700, 4096, 1024, 1)
    out = torch.empty(700 * (1 << 23), dtype=torch.bfloat16, device=DEV).as_strided((700, 4096), (1 << 23, 1))
    assert torch.equal(kernels.gemm_mid(A, B, variant=192, out=out), kernels.gemm_mid(A, B, variant=64))


@pytest.mark.parametrize("M,N,K", [(768, 4096, 14336), (560, 16384, 2048), (1500, 6144, 4096)])
@pytest.mark.parametrize("kind", ["plain", "residual", "glu"])
def test_where_the_plan_takes_it(M, N, K, kind):
    assert kernels.frag_plan(M, N, K) == (("192", M, N), None)
    glu = kind == "glu"
    A, B, exp = _case(M, N, K, 8 if glu else 1)
    r = torch.randn(M, N, device=DEV).to(torch.bfloat16) if kind == "residual" else None
    run = dict(residual=r, epilogue=ops.EPI_SWIGLU8 if glu else ops.EPI_NONE, b_group=8 if glu else 1)
    assert torch.equal(ops.gemm_bt(A, B, shuffled=True, **run), kernels.gemm_mid(A, B, variant=192, **run))
