"""The divided tiles of gemm_mid's 128-row kernel: counts of the parts that are in, owners that hand a tile over, counts of ended
workgroups (the launch's number, which the 256-row kernel's ready flags hold)."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"
# tiles cut between two groups, between many, and between groups joined over the XCDs
SHAPES = [(300, 512, 4096), (1093, 4096, 1024), (2200, 2560, 1024), (44, 256, 8192)]


def _case(M, N, K, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    A = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    W = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    return A, ops.shuffle_weights(W), A.float() @ W.float().t()


def _close(out, exp):
    # one rounding to bf16 (2^-8 of the value); the fp32 sums are far below 1e-4
    return (out.float() - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4


def _launch(A, B, out, spin_limit):
    s = torch.cuda.current_stream().cuda_stream
    slabs, cnt = kernels._mid_workspace(A.device, s)
    M, K = A.shape
    kernels.native().gemm_mid(A.data_ptr(), K, B.data_ptr(), out.data_ptr(), out.stride(0), 0, 0, M, B.shape[0], K, 0,
                              slabs.data_ptr(), slabs.numel() * 4, cnt.data_ptr(), cnt.numel(), s, spin_limit=spin_limit)


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_a_launch_that_gave_up_leaves_nothing_for_the_next(M, N, K):
    """Owners that look once and go on (a kernel whose owners give up may write NaN over their tile); the launches after it take
    only their own partial tiles."""
    for seed in range(4):
        A, B, exp = _case(M, N, K, seed)
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        _launch(A, B, out, 0)
        assert (_close(out, exp) | out.isnan()).all()
        for other in range(2):
            A, B, exp = _case(M, N, K, 100 + 10 * seed + other)
            assert _close(ops.kernels.gemm_mid(A, B), exp).all()


def test_the_count_of_launches_may_wrap():
    A, B, exp = _case(*SHAPES[1], 0)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        ended = kernels._mid_workspace(A.device, s.cuda_stream)[0].view(torch.int32)[-256::32]
        s.wait_stream(torch.cuda.default_stream())
        grid = torch.cuda.get_device_properties(0).multi_processor_count & ~7
        assert (1 << 32) % grid == 0 and not ended.any()
        ended.fill_(-2 * (grid // 8))
        for i in range(5):
            assert _close(ops.kernels.gemm_mid(A, B), exp).all()
            assert (ended == (i - 1) * (grid // 8)).all()


def test_replays_go_on_counting():
    """A captured launch replayed between eager ones on its workspace."""
    (M, N, K), s = SHAPES[2], torch.cuda.Stream()
    cases = [_case(M, N, K, seed) for seed in range(3)]
    A, B = cases[0][0].clone(), cases[0][1].clone()
    with torch.cuda.stream(s):
        s.wait_stream(torch.cuda.default_stream())
        ops.kernels.gemm_mid(A, B)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            outs = [ops.kernels.gemm_mid(A, B) for _ in range(3)]
        for i in range(6):
            a, b, exp = cases[i % 3]
            A.copy_(a)
            B.copy_(b)
            g.replay()
            a2, b2, exp2 = cases[(i + 1) % 3]
            eager = ops.kernels.gemm_mid(a2, b2)
            s.synchronize()
            assert all(_close(o, exp).all() for o in outs) and _close(eager, exp2).all()


# tiles in equal parts, of unequal length, in groups joined over the XCDs, parts of one K-step; with parts in front of others of
# their group's range and without
HANDED = [(300, 512, 4096), (44, 256, 8192), (384, 4096, 4096), (4096, 256, 4096), (300, 6144, 4096), (2000, 6144, 4096),
          (1093, 4096, 14336), (1400, 6144, 1024), (2200, 2560, 1024), (1500, 5120, 128)]


def _run(A, B, out, spin_limit, s, res=None, epilogue=0, group=1):
    slabs, cnt = kernels._mid_workspace(A.device, s.cuda_stream)
    (M, K), N = A.shape, B.shape[0]
    kernels.native().gemm_mid(A.data_ptr(), K, B.data_ptr(), out.data_ptr(), out.stride(0), 0 if res is None else res.data_ptr(),
                              N, M, N, K, epilogue, slabs.data_ptr(), slabs.numel() * 4, cnt.data_ptr(), cnt.numel(),
                              s.cuda_stream, variant=64, b_group=group, spin_limit=spin_limit)
    return cnt


@pytest.mark.parametrize("M,N,K", HANDED)
@pytest.mark.parametrize("kind", ["plain", "residual", "glu"])
@pytest.mark.parametrize("busy", [False, True])
def test_owners_that_do_not_wait_hand_their_tiles_over(M, N, K, kind, busy):
    """An owner whose other parts are not in on the first look stores its own, and the last one in finishes the tile: the bits of a
    launch that waits, and no count left.  Busy: a product on another stream holds CUs, so workgroups are placed unevenly."""
    A, B, _ = _case(M, N, K, 1)
    group, epilogue, width = (8, ops.EPI_SWIGLU8, N // 2) if kind == "glu" else (1, 0, N)
    res = torch.randn(M, N, device=DEV).to(torch.bfloat16) if kind == "residual" else None
    s, other = torch.cuda.current_stream(), torch.cuda.Stream()
    exp = torch.empty(M, width, dtype=torch.bfloat16, device=DEV)
    _run(A, B, exp, 1 << 22, s, res, epilogue, group)
    X = torch.randn(2000, 2048, device=DEV).to(torch.bfloat16)
    Y = ops.shuffle_weights(torch.randn(4096, 2048, device=DEV).to(torch.bfloat16))
    other.wait_stream(s)
    for _ in range(8):
        out = torch.full_like(exp, 7.0)
        if busy:
            with torch.cuda.stream(other):
                for _ in range(4):
                    ops.kernels.gemm256(X, Y, shuffled=True)
        cnt = _run(A, B, out, 0, s, res, epilogue, group)
        assert torch.equal(out, exp) and exp.isfinite().all()
        assert not cnt.any()
    torch.cuda.synchronize()


@pytest.mark.parametrize("M,N,K", [(2000, 6144, 4096), (1093, 4096, 14336), (300, 6144, 4096)])
def test_two_streams(M, N, K):
    """Launches of two streams whose owners wait for workgroups that the other launch keeps from being placed."""
    A, B, _ = _case(M, N, K, 2)
    exp = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    _run(A, B, exp, 1 << 22, torch.cuda.current_stream())
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = [[torch.empty_like(exp) for _ in range(20)] for _ in streams]
    for s in streams:
        kernels._mid_workspace(A.device, s.cuda_stream)
    torch.cuda.synchronize()
    for pair in zip(*outs):
        for s, out in zip(streams, pair):
            _run(A, B, out, -1, s)
    torch.cuda.synchronize()
    assert all(torch.equal(out, exp) for each in outs for out in each)
