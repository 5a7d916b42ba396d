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
