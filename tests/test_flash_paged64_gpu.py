"""Causal prefill attention with heads of 64 over a paged cache against 64 bits, at the edges of tiles, blocks and waves."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


# one query, a wave's 32, a tile's 64 and a block's 128 with one more and one less; keys of earlier steps in whole tiles and
# not, more than the 128 tiles whose block ids lie in registers; a sequence without queries; heads that divide by the XCDs or not
@pytest.mark.parametrize("Hq,Hkv,lens,past,bs", [
    (32, 8, [1], 0, 64), (8, 8, [31, 32, 33], 0, 64), (3, 1, [63, 64, 65, 1], 0, 64), (6, 2, [127, 0, 128, 129], 0, 128),
    (32, 8, [300, 7], 64, 64), (16, 8, [257, 140], 5, 64), (2, 1, [200, 1, 64], 8200, 64), (4, 4, [130], 8129, 128),
    (64, 16, [385, 1000], 0, 64), (5, 5, [640], 131, 192)])
@pytest.mark.parametrize("strided", [False, True])
def test_against_64_bits(Hq, Hkv, lens, past, bs, strided):
    D, T = 64, sum(lens)
    g = torch.Generator(device=DEV).manual_seed(T + Hq + past)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    ctx = [n + past if n else 0 for n in lens]
    need = [-(-c // bs) for c in ctx]
    bt = torch.zeros(len(lens), max(need), dtype=torch.int32)
    for i, b in enumerate(torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).to(torch.int32).split(need)):
        bt[i, :len(b)] = b
    kc, vc = r(sum(need), Hkv, bs, D), r(sum(need), Hkv, bs, D)
    q = (r(T, Hq + 3, D) * 2)[:, 1:-2] if strided else r(T, Hq, D) * 2
    for i, c in enumerate(ctx):  # rows behind a context are never read
        if c % bs:
            kc[bt[i, need[i] - 1], :, c % bs:] = float("nan")
            vc[bt[i, need[i] - 1], :, c % bs:] = float("nan")
    cu = torch.tensor([0, *lens]).cumsum(0).to(torch.int32).to(DEV)
    out = torch.full((T + 1, Hq, D), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.flash_attention_paged(q, kc, vc, bt.to(DEV), cu, torch.tensor(ctx, dtype=torch.int32, device=DEV), max(lens), causal=True,
                              out=out[:T])
    assert (out[T] == 7.0).all()
    for b, (n, c) in enumerate(zip(lens, ctx)):
        if not n:
            continue
        k, v = (ref.gather_paged(x, bt[b].to(DEV), c).double().transpose(0, 1) for x in (kc, vc))
        at = slice(int(cu[b]), int(cu[b + 1]))
        mask = torch.arange(c, device=DEV)[None] > torch.arange(c - n, c, device=DEV)[:, None]
        for h in range(Hq):
            kh, vh = k[h // (Hq // Hkv)], v[h // (Hq // Hkv)]
            p = torch.softmax(((q[at, h].double() @ kh.t().contiguous()) * D ** -0.5).masked_fill(mask, float("-inf")), -1)
            most, exp = p @ vh.abs(), p @ vh
            # rounding of the probabilities and of the result: 2^-8 of sum |p v| and of the result
            assert ((out[at, h].double() - exp).abs() <= 2.0 ** -8 * (most + exp.abs()) + 1e-4).all()
