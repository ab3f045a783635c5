"""Which decode projections take the tiles of 64 weight rows."""
import pytest

from django_assistant_bot_amd.models.projections import FragmentProjections

WIDE = {1: 30, 16: 30, 17: 31, 32: 31, 33: 13, 64: 13}
NARROW = {30: 43, 31: 44, 13: 12}


@pytest.mark.parametrize("M", WIDE)
def test_narrow_tiles_keep_one_workgroup_a_cu_or_halve_the_slices(M):
    p = FragmentProjections.__new__(FragmentProjections)
    wide, narrow = WIDE[M], NARROW[WIDE[M]]
    # not gated, (N, K): slices that cannot be halved, 264-380 workgroups of 64 rows
    for N, K in ((1280, 8192), (1280, 14336), (2560, 1024), (4608, 512)):
        assert p._stream_choice("qkv", M, N, K)[0] == wide
    for N, K in ((1024, 8192), (2048, 2048), (4096, 4096), (6144, 4096), (3072, 8192), (10240, 4096)):
        cfg, s = p._stream_choice("qkv", M, N, K)
        assert cfg == narrow and N // 64 * s >= min(192, N // 4)
    # halved slices that leave a long K
    for N, K in ((8192, 28672), (6144, 14336), (12288, 8192)):
        assert p._stream_choice("down", M, N, K)[0] == (narrow if M <= 16 else wide)
    assert p._stream_choice("down", M, 4096, 14336)[0] == (narrow if M <= 32 else wide)
    for tiles in (4, 64, 128, 129, 172, 191, 224):
        assert p._stream_choice("gate_up", M, 128 * tiles, 4096) == \
            (narrow if tiles <= 128 else wide, p._stream_splits(128 * tiles, 4096, 64 if tiles <= 128 else 128))
    assert p._stream_choice("lm_head", M, 128256, 4096)[0] == (narrow if M <= 16 else wide)
    assert p._stream_choice("lm_head", M, 128256, 2048)[0] == wide


@pytest.mark.parametrize("M", [65, 128])
def test_gate_up_above_64_rows(M):
    p = FragmentProjections.__new__(FragmentProjections)
    for tiles, cfg in ((64, 9), (128, 9), (129, 10), (172, 10), (224, 20)):
        assert p._stream_choice("gate_up", M, 128 * tiles, 4096)[0] == cfg
    assert p._stream_choice("qkv", M, 4096, 4096)[0] == 10
