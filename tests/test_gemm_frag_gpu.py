"""gemm_frag (prompts' projections on fragment-layout weights) against an fp64 product: every tile at its edges, its K-slices, the
sizes that the plan gives it, and a prefill that runs on it."""
import dataclasses

import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.models import AttnMeta, KVCache, LlamaModel, decoder_config
from django_assistant_bot_amd.models.weights import random_decoder_weights
from django_assistant_bot_amd.ops import kernels

pytestmark = pytest.mark.gpu
DEV = "cuda"
TILES = [(32, 64), (64, 64), (96, 64), (64, 128), (128, 128), (192, 128), (128, 256)]


def _operands(M, N, K, grp=1, pad=8):
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    A = torch.randn(M, K + pad, device=DEV, generator=g).to(torch.bfloat16)[:, :K]
    W = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    return A, W, ops.shuffle_weights(W, grp), g


# rows: one, a tile less one, tiles and one; columns: less than a tile, ragged; K-tiles: fewer than the groups of waves or the
# ring, uneven shares of the groups, many
@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("rows,N,K", [(0, 128, 64), (-1, 384, 192), (1, 640, 320), (2, 1152, 1024)])
@pytest.mark.parametrize("kind", ["plain", "residual", "glu", "glu_bias"])
def test_every_tile(tile, rows, N, K, kind):
    bm = TILES[tile][0]
    M = {0: 1, -1: bm - 1, 1: bm + 1, 2: 3 * bm + 17}[rows]
    glu = kind.startswith("glu")
    A, W, B, g = _operands(M, N, K, 8 if glu or rows == 1 else 1)
    r = torch.randn(M, N + 8, device=DEV, generator=g).to(torch.bfloat16)[:, :N] if kind == "residual" else None
    gb = torch.randn(N, device=DEV, generator=g) if kind == "glu_bias" else None
    n_out = N // 2 if glu else N
    wide = torch.full((M + 1, n_out + 8), 7.0, dtype=torch.bfloat16, device=DEV)
    got = ops.gemm_frag(A, B, residual=r, epilogue=ops.EPI_SWIGLU8 if glu else ops.EPI_NONE, out=wide[:M, :n_out], glu_bias=gb,
                        b_group=8 if glu or rows == 1 else 1, tile=tile).double()
    exp = A.double() @ W.double().t()
    if glu:
        v = exp.view(M, N // 16, 2, 8)
        if gb is not None:
            v = v + gb.double().view(2, N // 16, 8).transpose(0, 1)
        exp = (torch.nn.functional.silu(v[:, :, 0]) * v[:, :, 1]).reshape(M, n_out)
    # one rounding to bf16 (2^-8), a second with the residual; fp32 sums of K products of size K^-1/2, and in the gate v_exp
    # / v_rcp to a few fp32 units: 1e-4 covers both at these K
    tol = 2.0 ** -8 * exp.abs() + 1e-4
    if r is not None:
        exp = exp + r.double()
        tol = tol + 2.0 ** -8 * exp.abs()
    assert ((got - exp).abs() <= tol).all()
    assert (wide[M:] == 7.0).all() and (wide[:, n_out:] == 7.0).all()


@pytest.mark.parametrize("tile", range(len(TILES)))
@pytest.mark.parametrize("K,S", [(128, 2), (448, 3), (1024, 5), (640, 8)])
def test_slices(tile, K, S):
    M, N = TILES[tile][0] + 5, 384
    A, W, B, _ = _operands(M, N, K)
    got = ops.gemm_frag(A, B, slices=S, tile=tile)
    cut = [K // 64 * i // S * 64 for i in range(S + 1)]
    for i in range(S):
        exp = A[:, cut[i]:cut[i + 1]].double() @ W[:, cut[i]:cut[i + 1]].double().t()
        assert (got[i].double() - exp).abs().max() <= 1e-4  # fp32 sums


def test_what_is_refused():
    A, _, B, _ = _operands(40, 256, 128)
    out = torch.empty(40, 256, dtype=torch.bfloat16, device=DEV)
    for bad in (dict(slices=3), dict(slices=2, out=out), dict(slices=2, residual=out), dict(epilogue=ops.EPI_GELU), dict(out=out[:, :128])):
        with pytest.raises((ValueError, RuntimeError)):
            ops.gemm_frag(A, B, **bad)


@pytest.mark.parametrize("M,N,K", [(65, 1024, 1024), (260, 2048, 2048), (515, 3072, 2048), (140, 28672, 1024), (1093, 1024, 4096)])
@pytest.mark.parametrize("shift", [0, 4])
def test_sizes_taken_from_the_larger_kernels(M, N, K, shift):
    """Outputs 8 bytes off a 16-byte line, which gemm_frag's stores do not take, stay on those kernels, which do."""
    A, W, B, _ = _operands(M, N, K)
    assert kernels.frag_plan(M, N, K) == (("frag", M, N), None) and kernels.frag_plan(M, N, K, True, False)[0][0] != "frag"
    out = torch.empty(M * N + 8, dtype=torch.bfloat16, device=DEV)[shift:M * N + shift].view(M, N)
    assert kernels._frag_takes(A, B, out, None, None) == (shift == 0)
    got = ops.gemm_bt(A, B, shuffled=True, out=out).double()
    exp = A.double() @ W.double().t()
    assert ((got - exp).abs() <= 2.0 ** -8 * exp.abs() + 1e-4).all()


@pytest.mark.parametrize("lens", [(129,), (100, 99, 1), (300,), (400, 17)])
def test_prefill(lens, monkeypatch):
    """A model whose layers gemm_frag serves: against the same prefill without it and the fp32 reference."""
    cfg = dataclasses.replace(decoder_config("tiny-llama"), hidden=1024, intermediate=2048, heads=16, kv_heads=8, layers=2)
    w32 = random_decoder_weights(cfg, dtype=torch.float32, seed=5, interleave_mlp=True)
    m = LlamaModel(cfg, {k: v.to(torch.bfloat16) for k, v in w32.items()}, DEV, interleaved_mlp=True)
    T, bs = sum(lens), 64
    ids = torch.randint(0, cfg.vocab_size, (T,), generator=torch.Generator().manual_seed(T), dtype=torch.int32)
    blocks = [-(-n // bs) for n in lens]
    tables = torch.zeros((len(lens), max(blocks)), dtype=torch.int32)
    slots, pos, at = [], [], 0
    for i, (n, b) in enumerate(zip(lens, blocks)):
        tables[i, :b] = torch.arange(at, at + b)
        slots.append(torch.arange(n) + at * bs)
        pos.append(torch.arange(n, dtype=torch.int32))
        at += b

    def prefill(model, dev, dtype):
        kv = KVCache(cfg.layers, at, cfg.kv_heads, bs, cfg.head_dim, dev, dtype=dtype)
        meta = AttnMeta(decode=False, positions=torch.cat(pos).to(dev), slots=torch.cat(slots).to(dev),
                        block_tables=tables.to(dev), ctx_lens=torch.tensor(lens, dtype=torch.int32, device=dev),
                        cu_q=torch.tensor([0, *lens], dtype=torch.int32).cumsum(0, dtype=torch.int32).to(dev), max_q=max(lens))
        return model.forward(ids.to(dev), meta, kv)

    calls, orig = [], kernels.gemm_frag
    spy = lambda *a, **k: calls.append(k.get("slices", 0)) or orig(*a, **k)  # noqa: E731
    monkeypatch.setattr(kernels, "gemm_frag", spy)
    monkeypatch.setattr(ops, "gemm_frag", spy)
    got = prefill(m, DEV, torch.bfloat16)
    assert len(calls) >= 3 * cfg.layers  # qkv, o and down at least
    monkeypatch.setattr(kernels, "frag_plan", lambda M, N, K, cols=True, frag=True: kernels._frag_plan(M, N, K, cols, False)[0])
    monkeypatch.setattr(ops, "frag_slices", lambda M, N, K: 0)
    del calls[:]
    other = prefill(m, DEV, torch.bfloat16)
    assert not calls
    torch.testing.assert_close(got.float(), other.float(), atol=6e-2, rtol=5e-2)
    ref = LlamaModel(cfg, {k: v.bfloat16().float() for k, v in w32.items()}, "cpu", interleaved_mlp=True)
    assert (got.float().cpu() - prefill(ref, "cpu", torch.float32)).abs().max().item() < 0.15
