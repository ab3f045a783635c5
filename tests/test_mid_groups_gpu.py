"""gemm_mid on fewer groups than fit the chip, and prefill steps of up to 256 tokens on the streamed projections."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.models import AttnMeta, KVCache, LlamaModel, decoder_config
from django_assistant_bot_amd.models.weights import random_decoder_weights

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one to eight row tiles; equal parts of a tile, whole tiles, fewer groups than tiles, parts of unequal length
@pytest.mark.parametrize("M,N,K", [(1, 2048, 2048), (130, 2048, 2048), (257, 3072, 2048), (300, 512, 4096), (384, 4096, 4096),
                                   (777, 768, 3072), (1000, 3072, 2048), (500, 6144, 1024)])
@pytest.mark.parametrize("glu", [False, True])
def test_fewer_groups(M, N, K, glu):
    tm = -(-M // 128)
    assert 0 < ops.kernels.native().gemm_mid_groups(M, N, K) < 8 * (32 // tm)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    A = torch.randn(M, K, device=DEV, generator=g).to(torch.bfloat16)
    W = (torch.randn(N, K, device=DEV, generator=g) * K ** -0.5).to(torch.bfloat16)
    B = ops.shuffle_weights(W, 8 if glu else 1)
    res = None if glu else torch.randn(M, N, device=DEV, generator=g).to(torch.bfloat16)
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
    first = None
    for _ in range(3):  # the ready flags are down again after each launch
        out = ops.kernels.gemm_mid(A, B, residual=res, epilogue=ops.EPI_SWIGLU8 if glu else ops.EPI_NONE, b_group=8 if glu else 1,
                                   variant=64)  # (the 128-row kernel, whatever the estimates say)
        assert ((out.float() - exp).abs() <= tol).all()
        first = out if first is None else first
        assert torch.equal(out, first)


@pytest.mark.parametrize("lens", [(130,), (100, 99, 1), (256,), (257,)])
def test_prefill_up_to_256_tokens_streams_with_fp32_slabs(lens, monkeypatch):
    """Against the prefill on the other GEMMs and the fp32 reference; the partial sums stay in 32 bits."""
    cfg = decoder_config("tiny-llama")
    w32 = random_decoder_weights(cfg, dtype=torch.float32, seed=3, interleave_mlp=True)
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
        return model.forward(ids.to(dev), meta, kv), kv

    dtypes, orig = [], ops.stream_gemm
    monkeypatch.setattr(ops, "stream_gemm", lambda *a, **k: dtypes.append(k.get("slab_dtype", torch.float32)) or orig(*a, **k))
    h_s, kv_s = prefill(m, DEV, torch.bfloat16)
    monkeypatch.setattr(ops, "stream_gemm", orig)
    assert bool(dtypes) == (T <= 256) and set(dtypes) <= {torch.float32}
    m.PREFILL_STREAM_MAX_M = 0
    h_g, kv_g = prefill(m, DEV, torch.bfloat16)
    torch.testing.assert_close(h_s.float(), h_g.float(), atol=6e-2, rtol=5e-2)
    torch.testing.assert_close(kv_s.k.float(), kv_g.k.float(), atol=6e-2, rtol=5e-2)
    ref = LlamaModel(cfg, {k: v.bfloat16().float() for k, v in w32.items()}, "cpu", interleaved_mlp=True)
    h_ref, _ = prefill(ref, "cpu", torch.float32)
    assert (h_s.float().cpu() - h_ref).abs().max().item() < 0.15
