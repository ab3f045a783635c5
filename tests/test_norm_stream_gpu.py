"""Projections with the RMS norm in front of them in one launch (norm_stream.hip) against the norm kernel and an fp64 product."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# slices shorter and longer than the weight ring (32 chunks of 32, 16 on 128 rows), not a multiple of it; columns past a
# norm wave's share and not; one to four rows
@pytest.mark.parametrize("N,K,splits,bn,grp", [(64, 256, 1, 64, 1), (128, 256, 8, 64, 8), (192, 1056, 1, 64, 1), (256, 2048, 4, 128, 8),
                                               (128, 2560, 1, 128, 1), (640, 4096, 2, 64, 1), (256, 4096, 1, 128, 8)])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
@pytest.mark.parametrize("S,dtype", [(1, torch.bfloat16), (2, torch.float32), (3, torch.bfloat16), (8, torch.bfloat16), (9, torch.float32)])
def test_norm_stream(N, K, splits, bn, grp, M, S, dtype):
    g = torch.Generator(device=DEV).manual_seed(N + K + M)

    def rand(*shape):
        return torch.randn(*shape, device=DEV, generator=g)

    x = (rand(S, M, K) * S ** -0.5).to(dtype)
    rows = x[0] if S == 1 else x
    res, gain = rand(M, K).to(torch.bfloat16), (1 + 0.1 * rand(K)).to(torch.bfloat16)
    W = (rand(N, K) * K ** -0.5).to(torch.bfloat16)
    frag = ops.shuffle_weights(W, grp)
    for residual in (res, None):
        h, new = ops.rmsnorm(rows, gain, 1e-5, residual=residual)
        exp = h.double() @ W.double().t()
        # the row's length is summed in another order (a rounding step of a normalised element, 2^-8 of it, on few of them):
        # 2^-8 of the product's terms in the root of their squares, and the rounding of what is stored
        tol = 2.0 ** -8 * ((h.double() ** 2) @ (W.double() ** 2).t()).sqrt() + 1e-5
        for sd in (torch.float32, torch.bfloat16):
            y, got = ops.norm_stream(rows, gain, 1e-5, residual, frag, splits=splits, bn=bn, slab_dtype=sd, w_group=grp)
            assert got is None if residual is None else torch.equal(got, new)
            part = y.double() if splits > 1 else y.double()[None]
            store = 0 if splits > 1 and sd == torch.float32 else 2.0 ** -8 * part.abs().sum(0)
            assert y.dtype == (sd if splits > 1 else torch.bfloat16)
            assert ((part.sum(0) - exp).abs() <= tol + store).all()
        if splits == 1:
            y, _ = ops.norm_stream(rows, gain, 1e-5, residual, frag, bn=bn, epilogue=ops.EPI_SWIGLU8, w_group=grp)
            v = exp.view(M, N // 16, 2, 8)
            gate, up = v[:, :, 0].reshape(M, -1), v[:, :, 1].reshape(M, -1)
            tg, tu = (t.reshape(M, -1) for t in (tol.view(M, N // 16, 2, 8)[:, :, 0], tol.view(M, N // 16, 2, 8)[:, :, 1]))
            act = torch.nn.functional.silu(gate) * up
            assert ((y.double() - act).abs() <= 2.0 ** -8 * act.abs() + 1.1 * tg * up.abs() + (gate.abs() + tg) * tu + 1e-5).all()


def test_what_is_refused():
    w = ops.shuffle_weights(torch.zeros(128, 4096, dtype=torch.bfloat16, device=DEV))
    g = torch.ones(4096, dtype=torch.bfloat16, device=DEV)
    for M, splits, bn in ((5, 1, 64), (1, 3, 64), (1, 1, 96)):
        assert not ops.norm_stream_ok(M, 128, 4096, splits, bn)
        with pytest.raises(Exception):
            ops.norm_stream(torch.zeros(M, 4096, dtype=torch.bfloat16, device=DEV), g, 1e-5, None, w, splits=splits, bn=bn)
    assert not ops.norm_stream_ok(1, 128, 8192, 1, 64) and not ops.norm_stream_ok(1, 128, 128, 1, 64)
