"""gemm_mid's kernel with tiles of 256 rows (variant 256) against an fp32 product."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"
# one row; full and ragged row tiles; one to fourteen column tiles an XCD, more tiles than groups among them; an odd number of pairs of
# K-steps; the largest M.  By what a group's range holds: whole tiles, a part of one, or (of unequal length) a part that is stored and
# then more, up to a part that it is the owner of
WHOLE = [(1093, 4096, 1024), (1300, 10240, 1152), (2200, 6144, 1024), (700, 28672, 1024), (4096, 2048, 2048)]
PARTS = [(1, 2048, 1024), (44, 2048, 8192), (256, 4096, 1024), (257, 6144, 3072)]
MIXED = [(1093, 4096, 14336), (700, 28672, 2048), (1430, 6144, 4096)]
SHAPES = PARTS + WHOLE + MIXED


def test_what_the_sizes_cover():
    for shapes, kind in ((WHOLE, "whole"), (PARTS, "parts"), (MIXED, "mixed")):
        for M, N, K in shapes:
            groups, kt = kernels.native().gemm_mid_wide_groups(M, N, K, 1) // 8, K // 128  # of an XCD; pairs of K-steps a tile
            q, r = divmod(N // 2048 * kt, groups)
            start = [j * q + min(j, r) for j in range(groups + 1)]
            if all(s % kt == 0 for s in start):
                assert kind == "whole"
            elif r == 0 and all(s // kt == (e - 1) // kt for s, e in zip(start, start[1:])):
                assert kind == "parts"
            else:
                assert kind == "mixed"
                assert any(s % kt and e % kt and e > (s // kt + 1) * kt for s, e in zip(start, start[1:]))


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
    first = None
    for _ in range(3):  # the ready flags are down again after each launch, and the order of the sums is fixed
        out = kernels.gemm_mid(A, B, variant=256, b_group=group)
        # one rounding to bf16 (2^-8 of the value); the fp32 sums are far below 1e-4
        assert ((out.float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4).all()
        first = out if first is None else first
        assert torch.equal(out, first)
    out = kernels.gemm_mid(A, B, residual=res, variant=256, b_group=group)
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
    out = kernels.gemm_mid(A, B, epilogue=epilogue, variant=256, b_group=8, glu_bias=b)
    # one rounding to bf16; the sums' 1e-4 of either factor times the other's size, at most 8 or so
    assert ((out.float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-3).all()


@pytest.mark.parametrize("M,N,K", [(300, 2048, 4096), (1093, 4096, 14336), (1430, 6144, 4096)])
def test_a_launch_that_gave_up_leaves_nothing_for_the_next(M, N, K):
    """Owners that look at a flag once write NaN over their tile; the launches behind take only their own partial tiles.  (Of 40
    launches each the one with the fewest gave up 9, 34 and 5 tiles.)"""
    s = torch.cuda.current_stream().cuda_stream
    A, B, exp = _case(M, N, K, 1)
    slabs, cnt = kernels._mid_workspace(A.device, s)
    for _ in range(3):
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        kernels.native().gemm_mid(A.data_ptr(), A.stride(0), B.data_ptr(), out.data_ptr(), N, 0, 0, M, N, K, 0, slabs.data_ptr(),
                                  slabs.numel() * 4, cnt.data_ptr(), cnt.numel(), s, variant=256, spin_limit=0)
        near = (out.float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4
        assert (near | out.isnan()).all() and out.isnan().any()
        for variant in (256, 64, 256):
            out = kernels.gemm_mid(A, B, variant=variant)
            assert ((out.float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4).all()


@pytest.mark.parametrize("M,N,K", [(700, 4096, 14336), (1000, 4096, 14336), (1093, 4096, 14336), (1200, 4096, 14336), (1700, 4096, 14336)])
def test_the_kernel_of_128_rows_where_the_estimates_are_near(M, N, K):
    """Unless its estimate is 13 % less the 256-row kernel is not taken: the sums of K keep their order."""
    wide = kernels.native().gemm_mid_wide_groups(M, N, K, 0) > 0
    assert wide == (M >= 1200)
    A, B, _ = _case(M, N, K, 1)
    assert torch.equal(kernels.gemm_mid(A, B), kernels.gemm_mid(A, B, variant=256 if wide else 64))


@pytest.mark.parametrize("stride,residual", [(1 << 23, False), (1 << 23, True), ((1 << 23) - 8, False)])
def test_output_rows_that_lie_far_apart(stride, residual):
    """256 rows of 2^23 elements are 4 GiB, past a buffer descriptor: the 128-row kernel takes them."""
    M, N, K = 700, 28672, 4096
    assert kernels.native().gemm_mid_wide_groups(M, N, K, 0)
    A, B, exp = _case(M, N, K, 1)
    out, res = torch.empty(M * stride, dtype=torch.bfloat16, device=DEV).as_strided((M, N), (stride, 1)), None
    out.fill_(7.0)
    if residual:
        res = torch.empty(M * stride, dtype=torch.bfloat16, device=DEV).as_strided((M, N), (stride, 1))
        res.normal_()
    got = kernels.gemm_mid(A, B, residual=res, out=out).float()
    tol = 2.0 ** -8 * exp.abs() + 1e-4  # one rounding to bf16, a second with the residual
    if residual:
        exp = exp + res.float()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((got - exp).abs() <= tol).all()


@pytest.mark.parametrize("M,N,K", [(1093, 4096, 14336), (700, 28672, 2048), (257, 6144, 3072)])
@pytest.mark.parametrize("variants", [(256, 256), (256, 64)])
def test_two_streams(M, N, K, variants):
    """Two launches at a time, which share the CUs of each XCD: their owners wait for workgroups placed before them."""
    A, B, _ = _case(M, N, K, 1)
    exp = [kernels.gemm_mid(A, B, variant=v) for v in variants]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in streams:
        kernels._mid_workspace(A.device, s.cuda_stream)
    torch.cuda.synchronize()
    outs = [[], []]
    for _ in range(20):
        for s, v, out in zip(streams, variants, outs):
            with torch.cuda.stream(s):
                out.append(kernels.gemm_mid(A, B, variant=v))
    torch.cuda.synchronize()
    assert all(torch.equal(o, e) for out, e in zip(outs, exp) for o in out)
