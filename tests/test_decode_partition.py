"""Keys of a decode attention partition: halved where several are combined anyway and every half finds a CU."""
import pytest

from django_assistant_bot_amd.ops import native


@pytest.mark.parametrize("part", [256, 512])
def test_partitions_are_halved_inside_one_round_of_the_combine(part):
    keys = native().decode_partition
    half = part // 2
    for longest, items, parts, exp in (
            (1, 8, 16, part), (half + 1, 8, 16, part), (part, 1, 16, part),  # one partition: written directly
            (part + 1, 8, 16, half), (4 * part, 8, 16, half), (2 * part, 48, 16, half),
            (4 * part + 1, 1, 64, part),  # nine halves: a second round
            (2 * part, 49, 16, part),  # 196 halves
            (2 * part, 8, 4, half), (2 * part, 8, 3, part)):  # what the workspace holds
        assert keys(part, longest, items, parts) == exp
    assert keys(1024, 4000, 1, 64) == 1024 and keys(384, 1000, 1, 64) == 384


@pytest.mark.parametrize("contexts,Hkv,parts", [
    ([1], 8, 16), ([1200] * 8, 8, 16), ([4000] * 9, 8, 16), ([2000, 400, 300] * 4, 8, 16), ([1700, 1000, 300, 600] * 5, 8, 16),
    ([2900, 3100, 2500, 3900] * 6, 8, 16), ([1000] * 32, 8, 16), ([700, 1500] * 16, 8, 16), ([513] * 200, 1, 16), ([900, 0, 5000] * 30, 2, 16),
    ([8000, 4000] * 16, 8, 16), ([30_000] * 3, 8, 60), ([100_000], 8, 200)])
@pytest.mark.parametrize("slots", [256, 512])
def test_partitions_find_a_slot_each(contexts, Hkv, parts, slots):
    """The smallest in whole 128 keys, from the halved or whole 512 on, of which as many workgroups hold every one; 4096 where
    none of up to that size does."""
    items, longest = len(contexts) * Hkv, max(contexts)
    count = lambda size: Hkv * sum(-(-c // size) for c in contexts)
    first = native().decode_partition(512, longest, items, parts)
    fits = [s for s in range(first, 4097, 128) if count(s) <= slots]
    assert native().decode_partition_fit(512, contexts, Hkv, parts, slots) == (fits[0] if fits else 4096)


def test_partitions_stay_where_the_workspace_or_the_items_end():
    fit = lambda *a: native().decode_partition_fit(*a, 256)
    assert fit(512, [3000] * 12, 8, 5) == 512  # (the workspace covers 2560 keys: larger partitions would cover more)
    assert fit(512, [3000] * 12, 8, 6) > 512
    assert fit(512, [3000] * 33, 8, 16) == 512 and fit(2048, [3000] * 40, 8, 16) == 2048  # above 256 items
