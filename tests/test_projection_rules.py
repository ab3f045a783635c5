"""Which kernel a projection takes."""
import pytest

from django_assistant_bot_amd.ops.kernels import small_tile


@pytest.mark.parametrize("M,N,K,tile", [(5300, 768, 768, 3), (5400, 768, 768, -1), (4000, 1024, 1024, -1), (3900, 1024, 1024, 3),
                                        (3066, 1536, 384, 3), (2048, 2304, 768, 3), (1600, 3072, 768, 3), (2200, 2304, 768, -1)])
def test_tall_projections_leave_the_64_x_64_tiles_earlier(M, N, K, tile):
    assert small_tile(M, N, K) == tile
