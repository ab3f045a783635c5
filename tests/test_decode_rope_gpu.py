"""Decode attention on the qkv projection's slabs (rotation and cache write inside) against the two launches, bit for bit."""
import pytest
import torch

from django_assistant_bot_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


# contexts at the edges of a sub-tile (32 keys), a block (64), a partition (512, halved for few items) and of the four waves'
# round; fewer and more slabs than are held; a padded row (no slot), a slot elsewhere than at the context's end
@pytest.mark.parametrize("D,Hq,Hkv,B", [(128, 32, 8, 1), (128, 32, 8, 8), (128, 12, 3, 9), (128, 5, 1, 40), (128, 32, 8, 32), (64, 32, 8, 6),
                                        (64, 32, 8, 48), (64, 2, 2, 130)])
@pytest.mark.parametrize("S,dtype", [(0, torch.bfloat16), (2, torch.bfloat16), (3, torch.float32), (4, torch.bfloat16),
                                     (8, torch.bfloat16), (4, torch.float32)])
def test_rope_inside_the_attention(D, Hq, Hkv, B, S, dtype):
    g = torch.Generator(device=DEV).manual_seed(D + B + S)
    bs, longest = 64, 1536
    n = longest // bs
    ctx = torch.randint(1, longest + 1, (B,), device=DEV, generator=g, dtype=torch.int32)
    edges = [1, 32, 33, 64, 65, 128, 129, 256, 512, 513, 1024, 1536]
    for i, e in enumerate(edges[: max(1, B - 2)]):
        ctx[-1 - i] = e
    tables = torch.randperm(B * n, device=DEV, generator=g).view(B, n).to(torch.int32)
    kc = torch.randn(B * n + 1, Hkv, bs, D, device=DEV, generator=g).to(torch.bfloat16)
    vc = torch.randn(kc.shape, device=DEV, generator=g).to(torch.bfloat16)
    pos = ctx - 1
    slots = tables[torch.arange(B, device=DEV), (pos // bs).long()].long() * bs + pos % bs
    if B > 2:
        slots[0], slots[1] = -1, B * n * bs + 5  # (the second: a block of nobody's table)
    W = (Hq + 2 * Hkv) * D
    qkv = torch.randn(B, W, device=DEV, generator=g).to(dtype) if S == 0 else (
        torch.randn(S, B, W, device=DEV, generator=g) * S ** -0.5).to(dtype)
    turn = torch.arange(longest, device=DEV)[:, None] * 10000.0 ** (-torch.arange(0, D, 2, device=DEV) / D)
    cs = torch.stack([turn.cos(), turn.sin()], -1).contiguous()
    order = torch.argsort(ctx, descending=True).to(torch.int32)
    ws = ops.DecodeWorkspace(B, Hq, D, -(-longest // 256), DEV)
    for part, o in ((512, order), (256, None), (2048, order)):
        assert ops.decode_rope_ok(B, Hkv, D, part)
        k1, v1, k2, v2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
        q = ops.rope_kv_write(qkv, pos, cs, k1, v1, slots, Hq, Hkv, D)
        exp = ops.paged_decode(q, k1, v1, tables, ctx, part, ws, order=o)
        for _ in range(2):  # (again: the new token's row is there already)
            got = ops.paged_decode_rope(qkv, pos, cs, k2, v2, slots, Hq, tables, ctx, part, ws, order=o)
            assert torch.equal(got, exp) and torch.equal(k1, k2) and torch.equal(v1, v2)
    assert not ws.cnt.any()


def test_rotation_on_two_slots_above_a_workgroup_a_cu():
    """320 items in whole contexts: the rotation inside takes two slots and two rounds, the two launches one slot."""
    B, Hq, Hkv, D, bs, part = 40, 16, 8, 128, 64, 2048
    g = torch.Generator(device=DEV).manual_seed(0)
    ctx = torch.randint(1, 2048, (B,), device=DEV, generator=g, dtype=torch.int32)
    ctx[:4] = torch.tensor([2048, 1, 128, 2047])
    tables = torch.randperm(B * 32, device=DEV, generator=g).view(B, 32).to(torch.int32)
    k1, v1 = (torch.randn(B * 32, Hkv, bs, D, device=DEV, generator=g).to(torch.bfloat16) for _ in range(2))
    k2, v2, pos = k1.clone(), v1.clone(), ctx - 1
    slots = tables[torch.arange(B, device=DEV), (pos // bs).long()].long() * bs + pos % bs
    qkv = torch.randn(4, B, (Hq + 2 * Hkv) * D, device=DEV, generator=g).to(torch.bfloat16)
    cs = torch.rand(2048, D // 2, 2, device=DEV, generator=g)
    ws = ops.DecodeWorkspace(B, Hq, D, 4, DEV)
    for order in (None, torch.argsort(ctx, descending=True).to(torch.int32)):
        q = ops.rope_kv_write(qkv, pos, cs, k1, v1, slots, Hq, Hkv, D)
        exp = ops.paged_decode(q, k1, v1, tables, ctx, part, ws, order=order)
        got = ops.paged_decode_rope(qkv, pos, cs, k2, v2, slots, Hq, tables, ctx, part, ws, order=order)
        assert torch.equal(got, exp) and torch.equal(k1, k2) and torch.equal(v1, v2)


def test_rotation_in_longer_partitions_of_heads_of_64():
    """16 sequences whose partitions of 512 keys are more than two workgroups a CU: longer ones, against the two launches,
    which keep 512 (their sums meet in another order)."""
    B, Hq, Hkv, D, bs, part, n = 16, 32, 8, 64, 64, 512, 64
    g = torch.Generator(device=DEV).manual_seed(1)
    ctx = torch.randint(2000, n * bs, (B,), device=DEV, generator=g, dtype=torch.int32)
    ctx[:3] = torch.tensor([n * bs, 1, 3])
    tables = torch.randperm(B * n, device=DEV, generator=g).view(B, n).to(torch.int32)
    k1, v1 = (torch.randn(B * n, Hkv, bs, D, device=DEV, generator=g).to(torch.bfloat16) for _ in range(2))
    k2, v2, pos = k1.clone(), v1.clone(), ctx - 1
    slots = tables[torch.arange(B, device=DEV), (pos // bs).long()].long() * bs + pos % bs
    qkv = torch.randn(4, B, (Hq + 2 * Hkv) * D, device=DEV, generator=g).to(torch.bfloat16)
    cs = torch.rand(n * bs, D // 2, 2, device=DEV, generator=g)
    ws = ops.DecodeWorkspace(B, Hq, D, n * bs // 512, DEV)
    for order in (None, torch.argsort(ctx, descending=True).to(torch.int32)):
        q = ops.rope_kv_write(qkv, pos, cs, k1, v1, slots, Hq, Hkv, D)
        exp = ops.paged_decode(q, k1, v1, tables, ctx, part, ws, order=order).float()
        got = ops.paged_decode_rope(qkv, pos, cs, k2, v2, slots, Hq, tables, ctx, part, ws, order=order).float()
        assert torch.equal(k1, k2) and torch.equal(v1, v2)
        # both round the probabilities and the result to bf16, with other maxima: 2^-8 of sum |p v| (at most max |v|), twice
        assert ((got - exp).abs() <= 2 * 2.0 ** -8 * (exp.abs() + v1.abs().max().float())).all()
        assert (got - exp).norm() <= 2.0 ** -7 * exp.norm()
    assert not ws.cnt.any()


def test_what_is_refused():
    assert not ops.decode_rope_ok(33, 8, 128, 512) and not ops.decode_rope_ok(8, 8, 128, 16384)
    assert not ops.decode_rope_ok(49, 8, 64, 512) and not ops.decode_rope_ok(1, 8, 32, 512)
