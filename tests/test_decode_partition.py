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
