"""Which form the matrix-core launchers take, checked on the host: the rules are arithmetic on sizes."""
import numpy as np
import pytest

from dgpp_amd import _lib

FP8, MXFP8, NVFP4, MXFP4 = range(4)


def takes_tiles(fmt, m, n, k):
    return _lib.load().dgpp_bench_dense_takes_tiles(fmt, m, n, k)


def tile_rows(fmt, m, n, k, a4=0, beside=0, ws=0):
    return _lib.load().dgpp_bench_dense_tile_rows(fmt, a4, m, n, k, beside, ws)


@pytest.mark.parametrize("fmt", [FP8, MXFP8, NVFP4, MXFP4])
def test_dense_tiles_only_where_the_16_row_form_needs_more_than_a_round(fmt):
    """The line of the wide tiles alone: what a launch of NVFP4 activations follows, and from where on a plain one does not stream."""
    # few blocks of 128 x 128 leave the chip idle: measured 1.1 to 5 times slower than the 16-row form
    for m, n, k in [(65, 512, 6144), (100, 512, 4096), (100, 4096, 4096), (129, 1536, 2048), (256, 4096, 4096), (1000, 512, 8192),
                    (65, 12288, 4096), (300, 2048, 1024), (64, 131072, 4096), (1, 4096, 4096)]:
        assert not takes_tiles(fmt, m, n, k), (m, n, k)
        assert tile_rows(NVFP4, m, n, k, a4=1) == 0
    # measured 1.05 to 3.3 times faster
    for m, n, k in [(1000, 12288, 6144), (300, 6144, 4096), (1000, 2048, 2048), (128, 12288, 8192), (512, 4096, 1024), (4096, 512, 512),
                    (65, 17408, 4096)]:
        assert takes_tiles(fmt, m, n, k), (m, n, k)
        assert tile_rows(NVFP4, m, n, k, a4=1) == 128 and tile_rows(fmt, m, n, k) > 0


@pytest.mark.parametrize("fmt,m,n,k,rows", [
    # measured: 45 us in 128-row tiles from 65 to 600 rows; the narrow ones 26, 32; 25; 30; 16.4
    (FP8, 200, 4096, 4096, 32), (FP8, 400, 4096, 4096, 64), (MXFP8, 200, 4096, 4096, 32), (NVFP4, 400, 4096, 4096, 64),
    (MXFP4, 200, 4096, 4096, 32), (FP8, 150, 12288, 4096, 32), (MXFP4, 100, 12288, 4096, 32), (FP8, 1000, 1024, 2048, 32),
    (FP8, 1000, 12288, 6144, 128), (MXFP8, 64, 131072, 4096, 128),
    # streamed: few blocks, short walks past the fit (5.9 us against 7.1, 5.7 against 7.1), and up to 32 rows at any size
    (FP8, 100, 4096, 4096, 0), (FP8, 441, 802, 448, 0), (NVFP4, 256, 493, 512, 0), (NVFP4, 320, 587, 512, 0), (MXFP8, 33, 512, 1024, 0),
    (FP8, 32, 131072, 4096, 0), (FP8, 33, 131072, 4096, 64), (NVFP4, 1, 131072, 4096, 0)])
def test_dense_tiles_of_a_plain_launch(fmt, m, n, k, rows):
    assert tile_rows(fmt, m, n, k) == rows
    # beside another product only the wide ones, and over a workspace that takes the parts of k none
    assert tile_rows(fmt, m, n, k, beside=1) == (128 if m > 64 else 0)
    if k >= 2048 and -(-n // 64) * -(-m // 16) < 1024:
        assert tile_rows(fmt, m, n, k, ws=1) == 0
    else:
        assert tile_rows(fmt, m, n, k, ws=1) == rows


@pytest.mark.parametrize("fmt", [FP8, MXFP8, NVFP4, MXFP4])
def test_dense_tiles_never_take_a_launch_that_splits_over_a_workspace(fmt):
    """A launch with fewer than 1024 blocks of 64 x 16 and several K parts splits them over a workspace, which the caller
    (or the static entry point, which refuses what its array does not hold) provides for exactly these."""
    for n in (64, 512, 4096, 8256, 16384, 17408, 65536):
        for m in (17, 64, 65, 80, 129, 256, 257, 1024, 2000):
            if -(-n // 64) * -(-m // 16) < 1024:
                assert not any(takes_tiles(fmt, m, n, k) for k in (512, 2048, 4096, 17408)), (m, n)
                assert not any(tile_rows(fmt, m, n, k, ws=1) for k in (2048, 4096, 17408)), (m, n)


@pytest.mark.parametrize("fmt,a4,gate_up,k,below,above", [
    (FP8, 0, 0, 384, 48, 96), (FP8, 0, 0, 768, 32, 40), (FP8, 0, 0, 2048, 16, 24), (FP8, 0, 0, 4096, 12, 20),
    (FP8, 0, 1, 768, 16, 20), (FP8, 0, 1, 4096, 10, 14), (NVFP4, 0, 0, 512, 20, 28), (NVFP4, 0, 0, 1024, 16, 20),
    (NVFP4, 0, 1, 2048, 7, 10), (MXFP4, 0, 0, 512, 20, 28), (MXFP4, 0, 0, 1024, 12, 20), (MXFP4, 0, 1, 4096, 6, 8),
    (NVFP4, 1, 0, 512, 16, 24), (NVFP4, 1, 0, 2048, 12, 15), (NVFP4, 1, 0, 6144, 9, 16)])
@pytest.mark.parametrize("segs", [128, 288])
def test_grouped_tiles_by_rows_per_segment(fmt, a4, gate_up, k, below, above, segs):
    """The tiles are slower at `below` rows per segment and faster at `above` (measured), whatever the tokens among which
    they are shared out."""
    def takes(rows, tokens, long_segs=0):
        return _lib.load().dgpp_bench_grouped_takes_tiles(fmt, a4, gate_up, segs, k, tokens, rows * segs, long_segs)
    for top_k in (4, 10):
        assert not takes(below, max(129, below * segs // top_k))
        assert takes(above, max(129, above * segs // top_k))
        assert not takes(above, 128)
        assert takes(below, 129, 1)   # a shared expert's segment behind the others


@pytest.mark.parametrize("fmt,a4,gate_up,segs,n,k,narrow,wide", [
    (NVFP4, 0, 1, 128, 512, 4096, (1, 4, 16), (25, 44)), (NVFP4, 0, 0, 128, 4096, 512, (1, 4, 16, 25), (44,)),
    (NVFP4, 0, 1, 256, 2048, 6144, (2, 5, 12), (22,)), (MXFP4, 0, 1, 256, 1024, 4096, (1, 5, 12), (22,)),
    (FP8, 0, 1, 128, 768, 2048, (6,), (25,)), (FP8, 0, 0, 128, 2048, 768, (6, 16), (48,)), (FP8, 0, 1, 256, 2048, 7168, (4, 6), (14,)),
    (NVFP4, 1, 0, 128, 2048, 6144, (4, 16), (25,))])
def test_grouped_passes_of_32_rows_by_rows_per_segment(fmt, a4, gate_up, segs, n, k, narrow, wide):
    """Measured over whole layers, the 32-row passes are faster than the 16-row form and than the 128-row passes at `narrow` rows per
    segment, the 128-row passes at `wide`; the rows must be known, and segments of up to 128 rows take them at any number."""
    lib = _lib.load()
    def takes(rows, most=1000, total=None):
        return lib.dgpp_bench_grouped_takes_narrow(fmt, a4, gate_up, segs, n, k, most, rows * segs if total is None else total, 0)
    for rows in narrow:
        assert takes(rows) and not takes(rows, total=0)
    for rows in wide:
        assert not takes(rows) and takes(rows, most=128)
        assert lib.dgpp_bench_grouped_takes_tiles(fmt, a4, gate_up, segs, k, 1000, rows * segs, 0)


def test_grouped_passes_of_32_rows_not_where_segments_are_nearly_empty_or_alone_and_long():
    takes = _lib.load().dgpp_bench_grouped_takes_narrow
    assert not takes(FP8, 0, 1, 128, 768, 2048, 100, 3 * 128, 0) and not takes(NVFP4, 1, 0, 128, 2048, 6144, 100, 3 * 128, 0)
    assert not takes(NVFP4, 0, 1, 128, 512, 4096, 100, 127, 0) and takes(MXFP4, 0, 1, 256, 1024, 4096, 100, 8, 0)
    # a shared expert's own launch: while the 128-row passes would be one round of the chip
    assert takes(FP8, 0, 1, 1, 2048, 4096, 100, 100, 1) and takes(FP8, 0, 1, 1, 512, 4096, 3968, 3968, 1)
    assert not takes(FP8, 0, 1, 1, 512, 4096, 4096, 4096, 1) and not takes(FP8, 0, 1, 1, 17408, 4096, 129, 129, 1)


@pytest.mark.parametrize("fmt,a4,segs,wide,short", [(FP8, 0, 1, 14, 13), (FP8, 0, 8, 35, 34), (FP8, 0, 16, 64, 63), (NVFP4, 0, 1, 11, 10),
                                                    (NVFP4, 0, 8, 32, 31), (NVFP4, 0, 16, 56, 55), (NVFP4, 0, 63, 197, 196), (NVFP4, 0, 64, 64, 63),
                                                    (NVFP4, 1, 8, 35, 34), (MXFP4, 0, 1, 1, 0), (MXFP4, 0, 16, 1, 0)])
@pytest.mark.parametrize("gate_up", [0, 1])
def test_grouped_passes_of_32_rows_of_a_short_table(fmt, a4, segs, wide, short, gate_up):
    """Measured slower than the 16-row form in tables of few segments until each has some rows, but for MXFP4."""
    takes = lambda rows: _lib.load().dgpp_bench_grouped_takes_narrow(fmt, a4, gate_up, segs, 1024, 4096, 16, rows, 0)
    assert takes(wide) and not takes(short)


def test_grouped_tiles_without_the_rows_known():
    takes = _lib.load().dgpp_bench_grouped_takes_tiles
    assert takes(NVFP4, 0, 0, 1, 128, 129, 0, 0) and not takes(NVFP4, 0, 0, 1, 128, 128, 0, 0)   # one segment: a dense product
    # NVFP4 activations, four experts a token, 9 rows a segment: measured 1.1 to 1.4 times slower in the tiles
    assert not takes(NVFP4, 1, 0, 256, 6144, 512, 0, 0)
    assert takes(NVFP4, 1, 0, 256, 6144, 1024, 0, 0)


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


@pytest.mark.parametrize("cols", [32, 128])
@pytest.mark.parametrize("n_segs,row_tiles,total_rows", [
    (1, 4, 4096), (63, 8, 31), (64, 8, 1), (256, 32, 16384), (289, 64, 36864), (1024, 56, 655360), (32767, 1, 100), (32768, 1, 100),
    (65535, 2, 100000), (64, 262143, 1), (64, 262144, 1), (56, 262144, 8 * 128), (61, 262144, 1), (1, 1, 1 << 29), (1, 2, 1 << 30)])
def test_sorted_passes_hold_every_pass_within_what_they_count_and_what_a_launch_takes(cols, n_segs, row_tiles, total_rows):
    blocks = np.zeros(1, np.int64)
    items = _lib.load().dgpp_bench_tiled_plan(n_segs, 0, row_tiles, min(total_rows, 1 << 20), total_rows, cols, blocks.ctypes.data)
    least = n_segs + total_rows // cols                     # passes of any table of so many segments and rows, at most
    sorts = least >= 64 and n_segs < 1 << 15 and -(-least // 8) * 8 * row_tiles < 1 << 24
    assert (items > 0) == sorts
    if sorts:
        assert items >= least and items % 8 == 0 and blocks[0] == items * row_tiles and blocks[0] * 256 < 1 << 32


def test_the_streamed_shapes_hold_the_empty_parts_that_their_test_names():
    """K is cut in four parts of whole turns of four steps from 4096 elements on; FP4 steps are of 128."""
    from test_gpu_tiled import STREAM_SHAPES
    empty, with_part_tile = set(), set()
    for k in {k for _, _, k in STREAM_SHAPES if k >= 4096}:
        steps = -(-k // 128)
        if 3 * (-(-steps // 4) + 3 & ~3) >= steps:
            (with_part_tile if k % 128 else empty).add(k)
    assert empty >= {4352} and with_part_tile >= {4160, 4576}


@pytest.mark.parametrize("fmt,tokens,top_k,experts,hidden,inter,shared,launched,captured", [
    (NVFP4, 3, 8, 288, 4096, 512, 512, 2, 2), (NVFP4, 12, 8, 288, 4096, 512, 512, 1, 0), (NVFP4, 16, 8, 288, 4096, 512, 512, 2, 0),
    (NVFP4, 8, 8, 256, 4096, 2048, 2048, 2, 1), (NVFP4, 7, 8, 256, 4096, 2048, 2048, 2, 0), (NVFP4, 15, 4, 180, 6144, 768, 768, 1, 0),
    (NVFP4, 16, 4, 288, 6144, 512, 512, 0, 0), (NVFP4, 4, 4, 44, 7168, 2048, 2048, 0, 0),
    (MXFP4, 3, 8, 256, 4096, 1024, 1024, 2, 2), (MXFP4, 7, 8, 256, 4096, 1024, 1024, 1, 0), (MXFP4, 15, 8, 256, 4096, 1024, 1024, 1, 1),
    (MXFP4, 15, 8, 64, 2304, 576, 640, 1, 0), (MXFP4, 16, 8, 256, 2048, 512, 512, 0, 0),
    (FP8, 1, 8, 128, 2048, 768, 768, 2, 2), (FP8, 2, 8, 256, 6144, 1024, 1024, 1, 1), (FP8, 3, 8, 256, 6144, 1024, 1024, 1, 0),
    (FP8, 5, 8, 128, 2048, 768, 768, 2, 2), (FP8, 15, 8, 288, 4096, 512, 512, 1, 0)])
def test_merged_passes_of_a_decode_step(fmt, tokens, top_k, experts, hidden, inter, shared, launched, captured):
    """Measured faster than launches of their own, one after the other when launched and on two streams when captured."""
    def passes(graph, fits=1):
        return _lib.load().dgpp_bench_merged_passes(fmt, tokens, top_k, experts, hidden, inter, shared, graph, fits)
    assert (passes(0), passes(1)) == (launched, captured)
    # rows that have no merged form of down: gate and up alone, captured from three tokens on only where that is the rule anyway
    assert passes(0, 0) == min(launched, 1) * (tokens < 16)
    assert passes(1, 0) == (1 if tokens < 3 or captured == 1 else 0)


@pytest.mark.parametrize("m,n,k,form", [
    # through registers or 16 rows, measured faster than the ring: short walks, few rows of them, several rounds
    (20, 37178, 192, 0), (1, 131072, 1984, 0), (16, 65536, 1088, 0), (64, 40000, 128, 2), (163, 28995, 576, 2), (1113, 7514, 576, 3),
    (300, 4096, 960, 2), (1734, 4355, 1472, 3), (1538, 2164, 1024, 2), (160, 10571, 1088, 2), (147, 630, 2176, 0),
    # the ring: one round below sixteen steps, the chip's fullest XCD counted; any from there on
    (300, 4096, 1024, 6), (32, 22515, 1152, 7), (17, 65536, 1088, 7), (54, 8160, 1728, 4), (399, 7013, 1856, 8), (1, 16384, 4096, 5), (300, 4096, 6144, 6), (300, 6144, 4096, 7),
    (1000, 6144, 4096, 6), (267, 10658, 2688, 6), (33, 8192, 8192, 4),
    # and what no panel holds
    (1000, 6144, 6720, 6), (64, 8192, 8256, 0), (300, 8192, 8256, 2), (16, 4096, 6144, 0), (48, 4096, 6144, 0), (49, 4096, 6144, 4), (1, 1, 64, 0)])
def test_mxfp8_gemm_form(m, n, k, form):
    got = _lib.load().dgpp_bench_mxfp8_form(m, n, k)
    assert got == form
    assert got < 4 or 1024 <= k <= (6656 if got == 8 else 8192)
