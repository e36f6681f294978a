"""Which form the matrix-core launchers take, checked on the host: the rules are arithmetic on sizes."""
import pytest

from dgpp_amd import _lib

FP8, MXFP8, NVFP4, MXFP4 = range(4)


def takes_tiles(fmt, m, n, k):
    return _lib.load().dgpp_bench_dense_takes_tiles(fmt, m, n, k)


@pytest.mark.parametrize("fmt", [FP8, MXFP8, NVFP4, MXFP4])
def test_dense_tiles_only_where_the_16_row_form_needs_more_than_a_round(fmt):
    # few blocks of 128 x 128 leave the chip idle: measured 1.1 to 5 times slower than the 16-row form
    for m, n, k in [(65, 512, 6144), (100, 512, 4096), (100, 4096, 4096), (129, 1536, 2048), (256, 4096, 4096), (1000, 512, 8192),
                    (65, 12288, 4096), (300, 2048, 1024), (64, 131072, 4096), (1, 4096, 4096)]:
        assert not takes_tiles(fmt, m, n, k), (m, n, k)
    # measured 1.05 to 3.3 times faster
    for m, n, k in [(1000, 12288, 6144), (300, 6144, 4096), (1000, 2048, 2048), (128, 12288, 8192), (512, 4096, 1024), (4096, 512, 512),
                    (65, 17408, 4096)]:
        assert takes_tiles(fmt, m, n, k), (m, n, k)


@pytest.mark.parametrize("fmt", [FP8, MXFP8, NVFP4, MXFP4])
def test_dense_tiles_never_take_a_launch_that_splits_over_a_workspace(fmt):
    """A launch with fewer than 1024 blocks of 64 x 16 and several K parts splits them over a workspace, which the caller
    (or the static entry point, which refuses what its array does not hold) provides for exactly these."""
    for n in (64, 512, 4096, 8256, 16384, 17408, 65536):
        for m in (17, 64, 65, 80, 129, 256, 257, 1024, 2000):
            if -(-n // 64) * -(-m // 16) < 1024:
                assert not any(takes_tiles(fmt, m, n, k) for k in (512, 2048, 4096, 17408)), (m, n)
