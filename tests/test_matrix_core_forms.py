"""Which form the matrix-core launchers take, checked on the host: the rules are arithmetic on sizes."""
import numpy as np
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


def tiled_blocks(n_segs, long_segs, row_tiles, max_rows):
    """(segment, row tile, first pass, step) of each block of a grouped launch; block b runs on XCD b % 8."""
    place = np.zeros(4, np.int32)
    count = _lib.load().dgpp_bench_tiled_place(n_segs, long_segs, row_tiles, max_rows, -1, place.ctypes.data)
    out = []
    for b in range(count):
        _lib.load().dgpp_bench_tiled_place(n_segs, long_segs, row_tiles, max_rows, b, place.ctypes.data)
        out.append(tuple(int(v) for v in place))
    return out


@pytest.mark.parametrize("n_segs,long_segs,row_tiles,max_rows",
                         [(1, 0, 1, 129), (1, 1, 8, 4096), (1, 1, 12, 777), (1, 0, 136, 256), (3, 0, 5, 300), (8, 0, 4, 1000),
                          (9, 1, 16, 2048), (8, 1, 16, 640), (100, 0, 7, 129), (257, 1, 16, 4096), (31, 0, 33, 640)])
def test_tiled_grouped_blocks_cover_every_pass_once_and_spread_long_segments(n_segs, long_segs, row_tiles, max_rows):
    passes = -(-max_rows // 128)
    spread_from = 0 if n_segs < 8 else n_segs - long_segs
    seen, work = {}, [0] * 8
    for b, (seg, tile, slot, step) in enumerate(tiled_blocks(n_segs, long_segs, row_tiles, max_rows)):
        if seg < 0:
            continue
        assert 0 <= seg < n_segs and 0 <= tile < row_tiles and 0 <= slot < step
        for p in range(slot, passes, step):
            assert (seg, tile, p) not in seen
            seen[seg, tile, p] = b % 8
        if seg >= spread_from:
            work[b % 8] += 1
    assert len(seen) == n_segs * row_tiles * passes
    # a shared expert's segment, above all one that is alone in its launch, occupies all XCDs alike
    assert max(work) <= -(-sum(work) // 8)
    # the others stay on one XCD each, with their activation rows
    for seg in range(spread_from):
        assert {x for (s, _, _), x in seen.items() if s == seg} == {seg % 8}
