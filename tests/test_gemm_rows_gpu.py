"""Projections whose whole waves of tiles go to the 256 x 256 kernel and the rows behind them to the encoder's ring."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.models import BertEncoder, EncoderConfig, pack_sequences, random_encoder_weights
from django_assistant_bot_amd.ops import kernels

DEV = "cuda"
# rows behind the waves: one, less than a tile, more than one; (N, K, GELU, residual)
SIZES = [(3072, 768, True, False), (768, 768, False, True), (768, 3072, False, True), (2304, 768, False, False), (1024, 1024, False, True)]


def _rows(M, N, K, gelu, res):
    return ops.native().gemm256_rows(M, N, K, int(gelu), int(res))


@pytest.mark.parametrize("N,K,gelu,res", SIZES)
def test_rule(N, K, gelu, res):
    wave = 256 // (N // 256) * 256  # rows of one wave
    for M in (1, wave - 1, wave):
        assert _rows(M, N, K, gelu, res) == M
    for waves in (1, 2, 5, 12):
        whole = waves * 256 // (N // 256) * 256
        assert _rows(whole + 1, N, K, gelu, res) in ((whole, whole + 1) if waves == 12 else (whole,))
        assert _rows(whole + wave - 300, N, K, gelu, res) == whole + wave - 300  # nearly a wave
    M = 14 * 256 // (N // 256) * 256 + 1
    assert _rows(M, N, K, gelu, res) == M


def test_rule_leaves():
    assert _rows(24291, 768, 3072, True, True) == 24291  # a GELU with a residual: no such epilogue
    assert _rows(24291, 700, 3072, False, False) == 24291  # columns that are no whole tiles
    far = (128 << 20) // (2 * 768)  # from here on another tile order, worth more than the last wave
    whole = 12 * 256 // 9 * 256
    assert whole < far < whole + 300 and _rows(far + 1, 2304, 768, False, False) == far + 1


@pytest.mark.gpu
@pytest.mark.parametrize("N,K,gelu,res", SIZES)
@pytest.mark.parametrize("more", [1, 255, 700])
@pytest.mark.parametrize("bias", [True, False])
def test_rows_behind_the_waves(N, K, gelu, res, more, bias):
    whole = 256 // (N // 256) * 256
    M = whole + more
    assert _rows(M, N, K, gelu, res) == whole
    g = torch.Generator(device=DEV).manual_seed(M + N + K)

    def rnd(rows, cols, pad=0, scale=1.0):  # a view of wider rows: strides other than the width
        return (torch.randn(rows, cols + pad, device=DEV, generator=g) * scale).to(torch.bfloat16)[:, :cols]

    A, B, r = rnd(M, K, 8), rnd(N, K, 16, K ** -0.5), rnd(M, N, 8) if res else None
    b = rnd(1, N)[0].contiguous() if bias else None
    wide = torch.empty(M + 1, N + 8, dtype=torch.bfloat16, device=DEV).fill_(7.0)
    epi = ops.EPI_GELU if gelu else ops.EPI_NONE
    ops.gemm_bt(A, B, bias=b, residual=r, epilogue=epi, out=wide[:M, :N])
    assert (wide[M:] == 7.0).all() and (wide[:, N:] == 7.0).all()
    # both kernels sum K in one order
    one = kernels.gemm256(A, B, bias=b, residual=r, epilogue=epi)
    assert torch.equal(wide[:M, :N], one)
    exp = A[whole - 64:].double() @ B.double().t()
    exp = exp if b is None else exp + b.double()
    exp = torch.nn.functional.gelu(exp) if gelu else exp
    # a rounding to bf16 of the product and, with a residual, of the sum; fp32 sums of K products of size about K^-1/2
    tol = 2.0 ** -8 * exp.abs() + 1e-4
    if res:
        exp = exp + r[whole - 64:].double()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((one[whole - 64:].double() - exp).abs() <= tol).all()


@pytest.mark.gpu
def test_rows_that_the_ring_refuses_are_not_left_out(monkeypatch):
    M, N, K = 256 // 3 * 256 + 1, 768, 768
    assert _rows(M, N, K, False, False) == M - 1
    A, B = (torch.zeros(n, K, dtype=torch.bfloat16, device=DEV) for n in (M, N))
    monkeypatch.setattr(kernels, "_gemm_small_into", lambda *a: False)
    with pytest.raises(ValueError):
        ops.gemm_bt(A, B)


@pytest.mark.gpu
def test_the_encoders_projections_take_the_same_rows(monkeypatch):
    cfg = EncoderConfig("t", vocab_size=500, hidden=768, layers=1, heads=12, intermediate=3072)
    model = BertEncoder(cfg, random_encoder_weights(cfg, DEV, seed=1), DEV)
    lens = [500] * 44  # 86 row tiles of 256: 258 tiles of o and down, 1032 of up
    T = sum(lens)
    assert _rows(T, 768, 768, False, True) < T and _rows(T, 768, 3072, False, True) < T and _rows(T, 3072, 768, True, False) < T
    g = torch.Generator().manual_seed(3)
    args = pack_sequences([torch.randint(0, 500, (n,), generator=g).tolist() for n in lens], DEV)
    got = model.forward(*args)
    monkeypatch.setattr(ops, "encoder_forward", lambda *a: None)
    assert torch.isfinite(got.float()).all() and torch.equal(got, model.forward(*args))
