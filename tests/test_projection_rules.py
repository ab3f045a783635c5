"""Which kernel a projection takes."""
import pytest

from django_assistant_bot_amd.ops.kernels import native, small_tile


@pytest.mark.parametrize("M,N,K,tile", [(5300, 768, 768, 3), (5400, 768, 768, -1), (4000, 1024, 1024, -1), (3900, 1024, 1024, 3),
                                        (3066, 1536, 384, 3), (2048, 2304, 768, 3), (1600, 3072, 768, 3), (2200, 2304, 768, -1)])
def test_tall_projections_leave_the_64_x_64_tiles_earlier(M, N, K, tile):
    assert small_tile(M, N, K) == tile


# faster on the ring than on gemm256 or the 128 x 128 kernel; slower
@pytest.mark.parametrize("M,N,K,wins", [(6400, 768, 768, True), (5300, 1152, 384, True), (17400, 1152, 384, True), (25000, 640, 1280, True),
                                        (3200, 3072, 768, False), (4600, 2304, 768, False), (17500, 384, 1536, False),
                                        (11000, 640, 1280, False)])
def test_large_projections_on_the_ring_where_it_is_faster(M, N, K, wins):
    assert small_tile(M, N, K) == -1 and native().ring_wins(M, N, K, 0, 0) == wins
