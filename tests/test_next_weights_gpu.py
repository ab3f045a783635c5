"""Encoder launches of a few tokens give the same bits with workgroups behind them that read the next launch's weights."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
# bytes of the next weights: less than a load a thread, a part of 16 B, not a multiple of 128 (nothing is read), one load over a
# whole number of them, the usual 4.7 MB
NEXT = [128, 4096, 4100, 1 << 20, (1 << 20) + 128, 2 * 3072 * 768]


def _each(launch, out):
    """`launch(next, bytes)` without and with every size of the next weights (each on an allocation of its own)."""
    launch(0, 0)
    exp = out.clone()
    for n in NEXT:
        w = torch.randint(0, 256, ((n + 15) // 16 * 16,), dtype=torch.uint8, device=DEV)
        out.fill_(7.0)
        launch(w.data_ptr(), n)
        assert torch.equal(out, exp), n
    assert torch.isfinite(exp.float()).all()


def _r(*shape):
    return torch.randn(*shape, device=DEV).to(torch.bfloat16)


# grids that leave room for readers, that are no multiple of 8, and that leave none
@pytest.mark.parametrize("M,N,K", [(1, 768, 3072), (16, 64, 768), (19, 768, 3072), (19, 1000, 768), (64, 1024, 4096), (33, 1024, 1024)])
@pytest.mark.parametrize("tile", [0, 1, 6, 7, 8])
@pytest.mark.parametrize("gelu", [0, 1])
def test_split_tile(M, N, K, tile, gelu):
    A, B, b, r, out = _r(M, K), _r(N, K), _r(N), _r(M, N), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    s = torch.cuda.current_stream().cuda_stream
    _each(lambda w, n: ops.native().gemm_small(A.data_ptr(), K, B.data_ptr(), K, out.data_ptr(), N, b.data_ptr(),
                                               0 if gelu else r.data_ptr(), N, M, N, K, gelu, tile, s, next=w, next_bytes=n), out)


@pytest.mark.parametrize("M,N,K", [(1, 2304, 768), (19, 3072, 768), (32, 2304, 768), (40, 1024, 1024), (19, 4096, 1024)])
@pytest.mark.parametrize("tile", [0, 1])
def test_norm_and_projection(M, N, K, tile):
    x, g, o, B, b, out = _r(M, K), _r(K), _r(K), _r(N, K), _r(N), torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    rows, s = torch.empty_like(x), torch.cuda.current_stream().cuda_stream
    for gelu in (0, 1):
        _each(lambda w, n: ops.native().gemm_ln(x.data_ptr(), g.data_ptr(), o.data_ptr(), 1e-12, rows.data_ptr(), B.data_ptr(),
                                                b.data_ptr(), out.data_ptr(), M, N, K, gelu, tile, s, next=w, next_bytes=n), out)


@pytest.mark.parametrize("H,D,lens", [(768, 64, [19]), (768, 64, [40, 24]), (384, 32, [6]), (384, 32, [33, 30]), (1024, 64, [1]),
                                      (1024, 64, [32])])
def test_attention_and_projection(H, D, lens):
    T = sum(lens)
    qkv, w0, b, r, out = _r(T, 3 * H), _r(H, H), _r(H), _r(T, H), torch.empty(T, H, dtype=torch.bfloat16, device=DEV)
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(DEV)
    s = torch.cuda.current_stream().cuda_stream
    _each(lambda w, n: ops.native().gemm_attn(qkv.data_ptr(), cu.data_ptr(), len(lens), D, D ** -0.5, w0.data_ptr(), b.data_ptr(),
                                              r.data_ptr(), out.data_ptr(), T, H, s, next=w, next_bytes=n), out)


@pytest.mark.parametrize("rows,cols", [(1, 768), (8, 1024), (120, 768), (817, 1024), (3000, 768), (33, 384)])
@pytest.mark.parametrize("residual", [False, True])
def test_norm(rows, cols, residual):
    x, r, g, o, out = _r(rows, cols), _r(rows, cols), _r(cols), _r(cols), torch.empty(rows, cols, dtype=torch.bfloat16, device=DEV)
    s = torch.cuda.current_stream().cuda_stream
    _each(lambda w, n: ops.native().layernorm(out.data_ptr(), x.data_ptr(), r.data_ptr() if residual else 0, g.data_ptr(), o.data_ptr(),
                                              rows, cols, 1e-12, s, next=w, next_bytes=n, then=w, then_bytes=n // 2), out)


@pytest.mark.parametrize("rows,cols,S", [(1, 768, 2), (817, 768, 3), (600, 1024, 2), (2200, 384, 3)])
def test_norm_of_slabs(rows, cols, S):
    x, r, b, g, o = torch.randn(S, rows, cols, device=DEV), _r(rows, cols), _r(cols), _r(cols), _r(cols)
    out, s = torch.empty(rows, cols, dtype=torch.bfloat16, device=DEV), torch.cuda.current_stream().cuda_stream
    _each(lambda w, n: ops.native().layernorm_slabs(out.data_ptr(), x.data_ptr(), S, b.data_ptr(), r.data_ptr(), g.data_ptr(),
                                                    o.data_ptr(), rows, cols, 1e-12, s, next=w, next_bytes=n, then=w, then_bytes=n // 2), out)
