"""Which kernel the rows of a linear layer are sent to (host only)."""


def test_wide_layers_over_few_fp32_rows():
    """Beyond the second round of its workgroups the one-launch split is the slower one."""
    from tmq_amd import _capi
    one = _capi.load().tmq_fp32_rows_one_launch
    for M in (13, 16):
        assert [one(None, M, K, N) for K, N in ((40, 32768), (40, 32769), (1, 338116), (1024, 32768))] == [1, 0, 0, 1]
    for M in (9, 12):
        assert [one(None, M, K, N) for K, N in ((512, 65536), (512, 65537), (513, 32768), (513, 32769))] == [1, 0, 1, 0]
    for M in (5, 8):
        assert [one(None, M, K, N) for K, N in ((64, 131072), (64, 131073), (600, 32768), (600, 32769), (1025, 16384), (1025, 16385))] == \
            [1, 0, 1, 0, 1, 0]
    for M in (3, 4):
        assert [one(None, M, K, N) for K, N in ((8, 1 << 20), (1025, 16384), (1025, 16385))] == [1, 1, 0]
    assert one(None, 2, 1025, 16385) == 1


def test_long_reductions_on_the_same_tile_stay_with_mid():
    """Where ring.hip would take mid.hip's own tile, a long reduction is faster in mid.hip: whole weight blocks (K a multiple of
    2048), and single pairs from K = 2048 (16 x 32 tiles) or 2560 (32 x 64) on."""
    from tmq_amd import _capi
    kernel, SPLIT, RING = _capi.load().tmq_ternary_rows_kernel, 1, 16
    rows = lambda M, K, N: kernel(_capi.F16, M, K, N)
    for M, N in ((32, 4096), (64, 2048), (64, 4096), (82, 4160), (128, 4096), (256, 2048)):
        assert rows(M, 4096, N) == SPLIT, (M, N)
        assert rows(M, 1024, N) >= RING, (M, N)
    assert rows(80, 2048, 8192) == SPLIT and rows(48, 2048, 11008) >= RING          # one round of 64 x 64 tiles; two of 32 x 64
    assert [rows(17, K, 4096) >= RING for K in (1984, 2304)] == [True, False]       # 16 x 32
    assert [rows(128, K, 3072) >= RING for K in (2496, 2560)] == [True, False]      # 32 x 64
    assert [rows(621, K, 1536) >= RING for K in (640, 704)] == [True, False]        # 32 x 64, four wavefronts, two rounds
    assert rows(17, 64, 16) >= RING
    # fp32 row pairs: only whole weight blocks
    assert kernel(_capi.F32, 60, 3584, 4096) >= RING and kernel(_capi.F32, 64, 4096, 4096) == SPLIT
    assert kernel(_capi.F16, 16, 64, 64) < 0


def test_16_x_64_tiles_of_medium_reductions_are_not_taken():
    """(their cost is fitted too low there: 80 rows, 1792 -> 8192 9.5 us on them, 8.1 on 64 x 64)"""
    from tmq_amd import _capi
    kernel = _capi.load().tmq_ternary_rows_kernel
    for K in (1280, 1536, 1792):
        for M, N in ((80, 8192), (64, 11008), (256, 3072)):
            assert kernel(_capi.F16, M, K, N) != 16 + 6
