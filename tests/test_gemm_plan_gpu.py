"""Projections divided between gemm256 and gemm_mid (``frag_plan``) against an fp64 product."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops.kernels import frag_plan

pytestmark = pytest.mark.gpu
DEV = "cuda"


def test_plans_cover_the_product():
    for M in (1, 127, 128, 129, 255, 256, 257, 700, 1093, 2600, 4096, 4097, 4300, 9001):
        for N, K in ((256, 128), (4096, 4096), (6144, 4096), (28672, 4096), (4096, 14336), (2048, 2048)):
            for cols in (True, False):
                plan = frag_plan(M, N, K, cols)
                if plan is None:
                    continue
                (_, m, n), rest = plan
                if rest is None:
                    assert (m, n) == (M, N)
                else:
                    _, m2, n2 = rest
                    assert (m == m2 == M and n + n2 == N) or (n == n2 == N and m + m2 == M)
                    assert n % 256 == 0 and (m == M or m % 256 == 0) and (cols or n == N)


# (M, N, K): columns divided, rows divided, rows past gemm_mid's 4096, one kernel instead of the other
@pytest.mark.parametrize("M,N,K", [(700, 28672, 256), (1093, 28672, 512), (2570, 6144, 512), (3000, 6144, 256), (4300, 4096, 512),
                                   (2300, 4096, 512), (1700, 6144, 512)])
@pytest.mark.parametrize("kind", ["plain", "residual", "glu", "glu_bias"])
def test_planned_projection(M, N, K, kind):
    glu = kind.startswith("glu")
    grp = 8 if glu else 1
    g = torch.Generator(device=DEV).manual_seed(M + N)
    A = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    B = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    r = torch.randn(M, N, device=DEV, generator=g).to(torch.bfloat16) if kind == "residual" else None
    gb = torch.randn(N, device=DEV, generator=g) if kind == "glu_bias" else None
    got = ops.gemm_bt(A, ops.shuffle_weights(B, grp), residual=r, shuffled=True, b_group=grp, glu_bias=gb,
                      epilogue=ops.EPI_SWIGLU8 if glu else ops.EPI_NONE).double()
    exp = A.double() @ B.double().t()
    if glu:
        v = exp.view(M, N // 16, 2, 8)
        if gb is not None:
            v = v + gb.double().view(2, N // 16, 8).transpose(0, 1)
        exp = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
    # one rounding to bf16 (2^-8), a second with the residual; fp32 sums of K products of size K^-1/2, and in the gate
    # v_exp / v_rcp to a few fp32 units: 1e-4 covers both at these K
    tol = 2.0 ** -8 * exp.abs() + 1e-4
    if r is not None:
        exp = exp + r.double()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((got - exp).abs() <= tol).all()


# (M, N, K): nine to twenty-one row tiles whose whole groups leave slots over on every XCD; tiles cut between groups
# anywhere, whole tiles, one K-step a group, groups without one
JOINED = [(1093, 14336, 64), (1093, 4096, 14336), (1400, 6144, 1024), (2200, 2560, 1024), (2600, 6144, 192), (2200, 14336, 64),
          (2200, 3584, 64), (2600, 3072, 192), (1700, 768, 64)]


@pytest.mark.parametrize("M,N,K", JOINED)
@pytest.mark.parametrize("glu", [False, True])
def test_mid_groups_joined_over_xcds(M, N, K, glu):
    tm = -(-M // 128)
    assert ops.kernels.native().gemm_mid_groups(M, N, K) > 8 * (32 // tm)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    A = torch.randn(M, K, device="cuda", generator=g).to(torch.bfloat16)
    W = (torch.randn(N, K, device="cuda", generator=g) * K ** -0.5).to(torch.bfloat16)
    B = ops.shuffle_weights(W, 8 if glu else 1)
    res = None if glu else torch.randn(M, N, device="cuda", generator=g).to(torch.bfloat16)
    epi = ops.EPI_SWIGLU8 if glu else ops.EPI_NONE
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
    for _ in range(3):  # the counts are zero again after each launch
        out = ops.kernels.gemm_mid(A, B, residual=res, epilogue=epi, b_group=8 if glu else 1, variant=64)
        assert ((out.float() - exp).abs() <= tol).all()


# gemm_frag behind gemm256's whole waves: columns divided, rows divided, a single row, a gate's half columns and its bias
@pytest.mark.parametrize("M,N,K,kind,rows", [(700, 28672, 4096, "glu", False), (3500, 6144, 4096, "plain", False), (3500, 6144, 4096, "residual", False),
                                             (3100, 6144, 4096, "plain", True), (3100, 6144, 4096, "residual", True), (4097, 4096, 4096, "residual", True),
                                             (1200, 16384, 2048, "glu", True), (1200, 16384, 2048, "glu_bias", True)])
def test_gemm_frag_behind_the_waves(M, N, K, kind, rows):
    glu = kind.startswith("glu")
    first, rest = frag_plan(M, N, K, kind != "glu_bias")
    assert rest[0] == "frag" and (rest[2] == N) == rows and ops.kernels.corner_plan(M, N, K)[0] == 0
    grp, n_out = (8, N // 2) if glu else (1, N)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    A = torch.randn(M, K + 8, device=DEV, generator=g).to(torch.bfloat16)[:, :K]
    B = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    r = torch.randn(M, N + 16, device=DEV, generator=g).to(torch.bfloat16)[:, :N] if kind == "residual" else None
    gb = torch.randn(N, device=DEV, generator=g) if kind == "glu_bias" else None
    wide = torch.full((M + 1, n_out + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    got = ops.gemm_bt(A, ops.shuffle_weights(B, grp), residual=r, shuffled=True, b_group=grp, glu_bias=gb, out=wide[:M, :n_out],
                      epilogue=ops.EPI_SWIGLU8 if glu else ops.EPI_NONE).double()
    assert (wide[M:] == 7.0).all() and (wide[:, n_out:] == 7.0).all()
    exp = A.double() @ B.double().t()
    if glu:
        v = exp.view(M, N // 16, 2, 8)
        if gb is not None:
            v = v + gb.double().view(2, N // 16, 8).transpose(0, 1)
        exp = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, N // 2)
    # as ``test_planned_projection``; the gate's and the up projection's 1e-4 multiply the other's size, up to 8 or so
    tol = 2.0 ** -8 * exp.abs() + (1e-3 if glu else 1e-4)
    if r is not None:
        exp = exp + r.double()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((got - exp).abs() <= tol).all()
