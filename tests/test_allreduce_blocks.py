"""Ranks that wait in the all-reduce leave CUs of a device they share to the rank they wait for."""
import pytest

from django_assistant_bot_amd.ops import native
from django_assistant_bot_amd.parallel.custom_allreduce import blocks_for


@pytest.mark.parametrize("cus", [256, 304, 32])
@pytest.mark.parametrize("world", range(1, 9))
def test_waiting_ranks_leave_cus_free(world, cus):
    """All but one of the ranks spinning, a workgroup on a CU of its own: an eighth of the CUs is still empty, which takes a
    kernel whose workgroups fill a CU's registers or LDS."""
    blocks = blocks_for([("card", cus)] * world, native().ALLREDUCE_BLOCKS)
    assert 1 <= blocks <= native().ALLREDUCE_BLOCKS
    assert (world - 1) * blocks <= cus - cus // 8
    if cus == 256:
        assert blocks == (64, 64, 64, 64, 56, 44, 37, 32)[world - 1]


def test_ranks_on_devices_of_their_own_use_all_workgroups():
    most = native().ALLREDUCE_BLOCKS
    assert blocks_for([(d, 256) for d in range(8)], most) == most
    # every rank launches as many as the most crowded device allows
    mixed = [("a", 256)] * 7 + [("b", 256)]
    assert blocks_for(mixed, most) == blocks_for([("a", 256)] * 7, most) < most
