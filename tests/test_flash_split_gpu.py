"""Prefill attention with the keys of a query block split over two groups of waves, and the sizes around its rule."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


# odd and even numbers of 64-key tiles, a tile of one key, blocks of one query, a sequence without queries, keys of earlier
# steps (whole tiles and not), heads that divide by the XCDs and not; the last five are on the other side of the rule
@pytest.mark.parametrize("Hq,Hkv,lens,past", [
    (8, 2, [385], 0), (8, 2, [448], 0), (8, 2, [449], 0), (8, 2, [512, 1, 0, 130], 0), (6, 2, [513, 400], 0), (8, 2, [400], 64),
    (8, 2, [641], 333), (3, 1, [1093], 0), (8, 8, [385, 64, 70], 8200), (32, 8, [1093], 0), (32, 8, [2048], 0), (32, 8, [1000, 900], 7),
    (32, 8, [500, 385, 500], 0), (32, 8, [2049], 0), (8, 2, [384, 384], 0), (32, 8, [600, 600, 500], 0), (32, 8, [300] * 4, 0)])
@pytest.mark.parametrize("rope", [False, True])
def test_keys_in_two_groups(Hq, Hkv, lens, past, rope):
    D, bs, T = 128, 64, sum(lens)
    g = torch.Generator(device=DEV).manual_seed(T + Hq + past)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV).to(torch.bfloat16)  # noqa: E731
    ctx = [n + past if n else 0 for n in lens]
    need = [-(-c // bs) for c in ctx]
    bt = torch.zeros(len(lens), max(need), dtype=torch.int32)
    for i, b in enumerate(torch.randperm(sum(need), generator=torch.Generator().manual_seed(1)).to(torch.int32).split(need)):
        bt[i, :len(b)] = b
    q, kc, vc = r(T, Hq, D) * 2, r(sum(need), Hkv, bs, D), r(sum(need), Hkv, bs, D)
    cu = torch.tensor([0, *lens]).cumsum(0).to(torch.int32).to(DEV)
    ctxt = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    pos = torch.cat([torch.arange(c - n, c) for c, n in zip(ctx, lens)]).to(torch.int32).to(DEV)
    turn = torch.arange(max(ctx), device=DEV)[:, None] * 10000.0 ** (-torch.arange(0, D, 2, device=DEV) / D)
    cs = torch.stack([turn.cos(), turn.sin()], -1).contiguous()
    out = ops.flash_attention_paged(q, kc, vc, bt.to(DEV), cu, ctxt, max(lens), causal=True, rope=(pos, cs) if rope else None)
    qr = ref.rope_q(q, pos, cs) if rope else q
    for b, (n, c) in enumerate(zip(lens, ctx)):
        if not n:
            continue
        k, v = (ref.gather_paged(x, bt[b].to(DEV), c).double().transpose(0, 1) for x in (kc, vc))
        at = slice(int(cu[b]), int(cu[b + 1]))
        mask = torch.arange(c, device=DEV)[None] > torch.arange(c - n, c, device=DEV)[:, None]
        for h in range(Hq):
            kh, vh, qh = k[h // (Hq // Hkv)], v[h // (Hq // Hkv)], qr[at, h].double()
            s = ((qh @ kh.t().contiguous()) * D ** -0.5).masked_fill(mask, float("-inf"))
            p = torch.softmax(s, -1)
            # rounding of the probabilities and of the result: 2^-8 of sum |p v| and of the result.  The rotated q may round to
            # its other neighbour: 2^-8 of sum |q k| in a score, twice that of sum |p v|
            most, exp = p @ vh.abs(), p @ vh
            moved = 2.0 ** -8 * ((qh.abs() @ kh.abs().t().contiguous()) * D ** -0.5).masked_fill(mask, 0).amax(1, keepdim=True)
            bound = 2.0 ** -8 * (most + exp.abs()) + (2 * moved * most if rope else 0.0) + 1e-4
            assert ((out[at, h].double() - exp).abs() <= bound).all()


# either side of the rule with 32 heads: a workgroup a CU at most, one and a quarter, one and a half, two with blocks enough
@pytest.mark.parametrize("lens", [[500], [1093], [2000], [500, 500], [400] * 3, [450] * 3, [560, 560], [700, 700], [780, 780], [900, 900]])
def test_the_rule_costs_no_more_than_a_block_a_workgroup(lens, monkeypatch):
    """Keys in two groups for 256 to 384 blocks of four to six a sequence took up to 1.2 times as long as a block a workgroup."""
    Hq, Hkv, D, bs, B, layers = 32, 8, 128, 64, len(lens), 6
    n = -(-max(lens) // bs)
    caches = [torch.randn(2, B * n, Hkv, bs, D, device=DEV).to(torch.bfloat16) for _ in range(layers)]
    bt = torch.randperm(B * n).view(B, n).to(torch.int32).to(DEV)
    q = torch.randn(sum(lens), Hq, D, device=DEV).to(torch.bfloat16)
    cu, ctx = torch.tensor([0, *lens]).cumsum(0).to(torch.int32).to(DEV), torch.tensor(lens, dtype=torch.int32, device=DEV)

    def us():
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        torch.cuda.synchronize()
        a.record()
        for i in range(24):
            ops.flash_attention_paged(q, *caches[i % layers], bt, cu, ctx, max(lens), causal=True)
        b.record()
        b.synchronize()
        return a.elapsed_time(b) / 24 * 1e3
    taken, single = [], []
    for _ in range(8):  # in turn: the least of each
        monkeypatch.delenv("DAB_FLASH_PAIR", raising=False)
        taken.append(us())
        monkeypatch.setenv("DAB_FLASH_PAIR", "0")
        single.append(us())
    print(f"{lens}: {min(taken):.1f} us, a block a workgroup {min(single):.1f}")
    assert min(taken) <= 1.08 * min(single)
