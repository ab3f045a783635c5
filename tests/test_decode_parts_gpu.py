"""Partitions of the paged decode attention (halved for few items, combined eight at a time) against an fp64 softmax."""
import pytest
import torch

from django_assistant_bot_amd import ops
from django_assistant_bot_amd.ops import reference as ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


# halved: up to 192 items and a workspace that holds them (max_parts); 64 and 65 sequences: lengths held in lanes or not;
# 8 / 9 / 17 partitions: one, two and three rounds of the combine; above 64 items partitions doubled once, twice, up to
# 2048 keys with items left for a second and third round of 256 workgroups, and not where the workspace then covered more
@pytest.mark.parametrize("ctx,Hkv,max_parts", [([1], 8, 16), ([256, 257], 8, 16), ([2048], 2, 8), ([2049], 2, 9), ([2048], 2, 7),
                                               ([4200, 3], 1, 32), ([513] * 12, 8, 4), ([513] * 13, 2, 4), ([70] * 63 + [900], 1, 2),
                                               ([70] * 64 + [1100], 1, 3), ([1700, 600, 513, 512] * 4, 8, 4),
                                               ([2000, 1500, 90, 1] * 6, 8, 4), ([5000, 2049, 4100, 7] * 8, 8, 10),
                                               ([1500] * 16, 8, 2), ([2100] * 70, 3, 5)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("order", [False, True])
def test_decode_partitions(ctx, Hkv, max_parts, D, order):
    _check(ctx, Hkv, max_parts, D, order)


# two slots: partitions of as many keys as give every one a workgroup, and those alone walked: sequences without and with a
# second and third one in any place, none (a padded row), words of 64 sequences, contexts beyond the largest partition
@pytest.mark.parametrize("ctx,Hkv,max_parts", [([200, 2000, 10, 1100] * 3, 8, 4), ([4000, 100] * 5 + [4000], 8, 8), ([300] * 31 + [5000], 8, 10),
                                               ([600, 0, 1300, 513] * 16, 4, 4), ([900, 20, 30] * 66, 1, 4), ([30] * 255 + [2500], 1, 6),
                                               ([9000, 700] * 5, 8, 20), ([3000, 9000, 5000] * 10, 8, 18)])
@pytest.mark.parametrize("order", [False, True])
def test_partitions_that_find_a_workgroup_each(ctx, Hkv, max_parts, order):
    _check(ctx, Hkv, max_parts, 128, order)


def _check(ctx, Hkv, max_parts, D, order):
    g = torch.Generator(device=DEV).manual_seed(len(ctx) + Hkv)
    B, Hq, bs = len(ctx), 4 * Hkv, 64
    need = [-(-c // bs) for c in ctx]
    blocks = torch.randperm(sum(need), generator=torch.Generator().manual_seed(0)).to(torch.int32)
    bt = torch.zeros(B, max(need), dtype=torch.int32)
    for i, b in enumerate(blocks.split(need)):
        bt[i, :len(b)] = b
    kc, vc = (torch.randn(sum(need), Hkv, bs, D, device=DEV, generator=g).to(torch.bfloat16) for _ in range(2))
    q = torch.randn(B, Hq, D, device=DEV, generator=g).to(torch.bfloat16)
    ctxt = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    by_len = torch.argsort(-ctxt).to(torch.int32) if order else None
    ws = ops.DecodeWorkspace(B, Hq, D, max_parts, DEV)
    for _ in range(2):  # the arrival counters are zero again after a launch
        out = ops.paged_decode(q, kc, vc, bt.to(DEV), ctxt, 512, ws, order=by_len)
        for b, n in enumerate(ctx):
            if n == 0:
                continue
            n = min(n, 512 * max_parts)  # what the workspace's partitions cover
            k, v = (ref.gather_paged(c, bt[b].to(DEV), n).double().repeat_interleave(4, 1).transpose(0, 1) for c in (kc, vc))
            s = torch.matmul(k, q[b].double().unsqueeze(-1)).squeeze(-1) * D ** -0.5
            p = torch.softmax(s, -1)
            exp = torch.matmul(p.unsqueeze(1), v).squeeze(1)
            # probabilities and result rounded to bf16: 2^-8 of the sum of |p v| and of the result
            bound = 2.0 ** -8 * (torch.matmul(p.unsqueeze(1), v.abs()).squeeze(1) + exp.abs()) + 1e-4
            assert ((out[b].double() - exp).abs() <= bound).all()
    assert not ws.cnt.any()
