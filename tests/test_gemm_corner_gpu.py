"""Whole waves of 256 x 256 tiles without the end of the last row of them, and gemm_frag's corner behind (``corner_plan``)."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops import kernels

DEV = "cuda"


# quicker so by measurement; not, or nothing of a last row is left over (rows, N, K)
@pytest.mark.parametrize("M,N,K,takes", [(1093, 28672, 4096, True), (640, 28672, 4096, False), (1600, 28672, 4096, True), (5701, 28672, 4096, True), (2760, 6144, 4096, True), (2565, 6144, 4096, True),
                                         (5626, 3072, 2048, True), (2880, 28672, 4096, False), (1024, 28672, 4096, False),
                                         (256, 28672, 4096, False), (700, 4096, 4096, False), (1093, 16384, 2048, False), (1093, 28672, 4000, False)])
def test_plan(M, N, K, takes):
    tail, us = kernels.corner_plan(M, N, K)
    assert (tail > 0) == takes == (us is not None)
    if takes:
        tm, tn = -(-M // 256), N // 256
        assert tail < tn and ((tm - 1) * tn + tail) % 256 == 0
        assert us < kernels._frag_plan(M, N, K, True, True)[1]


def _operands(M, N, K, glu, res):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    A = torch.randn(M, K + 8, device=DEV, generator=g).to(torch.bfloat16)[:, :K]
    W = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    r = torch.randn(M, N + 16, device=DEV, generator=g).to(torch.bfloat16)[:, :N] if res else None
    return A, W, ops.shuffle_weights(W, 8 if glu else 1), r


def _check(got, A, W, r, glu):
    exp = A.double() @ W.double().t()
    if glu:
        v = exp.view(len(A), -1, 2, 8)
        exp = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(len(A), -1)
    # one rounding to bf16 (2^-8), a second with the residual; fp32 sums of K products of size K^-1/2, and in the gate
    # v_exp / v_rcp to a few fp32 units
    tol = 2.0 ** -8 * exp.abs() + 1e-4
    if r is not None:
        exp = exp + r.double()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((got.double() - exp).abs() <= tol).all()


# the last row of one, some and all but one of its tiles; of one row and of 256; one group of row tiles and several; blocks of columns
@pytest.mark.gpu
@pytest.mark.parametrize("M,N,tail", [(257, 512, 1), (513, 768, 2), (1093, 1024, 1), (1536, 2560, 9), (1800, 256 * 70, 33), (300, 256 * 66, 65)])
@pytest.mark.parametrize("glu,res", [(True, False), (False, True), (False, False)])
def test_last_row_of_tiles(M, N, tail, glu, res):
    K = 256
    A, W, B, r = _operands(M, N, K, glu, res)
    epi, per, m = (ops.EPI_SWIGLU8, 2, (M - 1) // 256 * 256) if glu else (ops.EPI_NONE, 1, (M - 1) // 256 * 256)
    wide = torch.full((M + 1, N // per + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    out = wide[:M, :N // per]
    kernels._gemm256_into(A, B, out, None, r, epi, True, 8 if glu else 1, tail)
    assert (out[m:, 256 * tail // per:] == 7.0).all() and (wide[M:] == 7.0).all() and (wide[:, N // per:] == 7.0).all()
    kernels._run_corner(tail, A, B, out, r, epi, 8 if glu else 1)
    _check(out, A, W, r, glu)
    assert (wide[M:] == 7.0).all() and (wide[:, N // per:] == 7.0).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K,glu,res", [(1093, 28672, 4096, True, False), (2760, 6144, 4096, False, False), (2760, 6144, 4096, False, True)])
def test_sizes_taken(M, N, K, glu, res, monkeypatch):
    assert kernels.corner_plan(M, N, K)[0]
    A, W, B, r = _operands(M, N, K, glu, res)
    calls, orig = [], kernels._run_corner
    monkeypatch.setattr(kernels, "_run_corner", lambda *a: calls.append(1) or orig(*a))
    epi, per = (ops.EPI_SWIGLU8, 2) if glu else (ops.EPI_NONE, 1)
    kw = dict(residual=r, shuffled=True, b_group=8 if glu else 1, epilogue=epi)
    _check(ops.gemm_bt(A, B, **kw), A, W, r, glu)
    assert calls
    # outputs 8 bytes off a 16-byte line, which gemm_frag's stores do not take, and biases of the gate
    out = torch.empty(M * (N // per) + 8, dtype=torch.bfloat16, device=DEV)[4:-4].view(M, N // per)
    _check(ops.gemm_bt(A, B, out=out, **kw), A, W, r, glu)
    if glu:
        _check(ops.gemm_bt(A, B, glu_bias=torch.zeros(N, device=DEV), **kw), A, W, r, glu)
    assert len(calls) == 1


@pytest.mark.gpu
def test_what_is_refused():
    A, _, B, _ = _operands(257, 512, 256, False, False)
    out = torch.empty(257, 512, dtype=torch.bfloat16, device=DEV)
    for rows, tail in ((257, 3), (257, -1), (256, 1)):
        with pytest.raises((ValueError, RuntimeError)):
            kernels._gemm256_into(A[:rows], B, out[:rows], None, None, ops.EPI_NONE, True, 1, tail)
