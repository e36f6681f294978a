"""The MXFP8 GEMM's forms for many activation rows against its 16-row form, bit for bit: all add the same steps of the
same chains in the same order, and the 16-row form is held to the oracle in test_gpu_mxfp8.py. Sizes at the edges of the
tiles of 32, 64 and 128 rows, k of a part of a step, of fewer steps than chains and of several steps a chain, scale
rows that are whole words and not, and a scale pointer that is no word's. Bench switch 15 pins the form."""
import numpy as np
import pytest

import mxfp8_data as md
from dgpp_amd import _lib, launch as L
from gpu_util import dev, dev_empty, host, sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1, 1, 64), (65, 63, 128), (64, 64, 192), (129, 130, 1088), (200, 128, 2048), (128, 257, 6144),
                                   (333, 200, 2112)])
def test_tiled_is_bitwise_the_16_row_form(gpu, m, n, k):
    a, a_s, w, w_s = md.gemm_case(m, n, k, 3)
    a_d, as_d, w_d, ws_d = dev(a), dev(a_s), dev(w), dev(w_s)
    shifted = dev(np.concatenate([np.zeros(1, np.uint8), a_s.reshape(-1)]))
    out, outh = dev_empty((m, n + 7), np.float32), dev_empty((m, n + 4), np.uint16)
    want = None
    for form in (1, 2, 3, 4, 0):
        for scales in (as_d, shifted[1:]):
            out.fill_(-1)
            outh.fill_(0x55)
            _lib.load().dgpp_tune_set(15, form)
            try:
                L.launch_mxfp8_gemm_f32(a_d, scales, w_d, ws_d, out, m, n, k, None, n + 7)
                L.launch_mxfp8_gemm_bf16(a_d, scales, w_d, ws_d, outh, m, n, k, None, n + 4)
            finally:
                _lib.load().dgpp_tune_set(15, 0)
            sync()
            got = host(out).view(np.uint32).copy(), host(outh).copy()
            want = want or got
            for x, y in zip(want, got):
                assert np.array_equal(x, y), (form, m, n, k)


@pytest.mark.parametrize("k", [192, 1088, 2112])
def test_non_finite_codes_and_scales_reach_the_same_outputs(gpu, k):
    """NaN codes and scales in the first, an inner and the last block of some rows of either operand; k is no multiple of a
    step, so the lanes past it read bytes that are their row's own."""
    m, n = 70, 66
    a, a_s, w, w_s = md.gemm_case(m, n, k, 4)
    a[2, 0], a[30, k - 1], w[7, k // 2], w[65, 0] = 0x7F, 0xFF, 0x7F, 0xFF
    a_s[11, 0] = a_s[69, -1] = w_s[20, -1] = w_s[33, 1] = 0xFF
    nan_rows, nan_cols = [2, 11, 30, 69], [7, 20, 33, 65]
    ops = [dev(v) for v in (a, a_s, w, w_s)]
    out = dev_empty((m, n), np.float32)
    want = None
    for form in (1, 2, 3, 4):
        out.fill_(-1)
        before = _lib.load().dgpp_bench_tiled_launches()
        _lib.load().dgpp_tune_set(15, form)
        try:
            L.launch_mxfp8_gemm_f32(*ops, out, m, n, k)
        finally:
            _lib.load().dgpp_tune_set(15, 0)
        sync()
        assert _lib.load().dgpp_bench_tiled_launches() - before == (form > 1)
        got = host(out).copy()
        want = got if want is None else want
        nan = np.isnan(got)
        expected = np.zeros((m, n), bool)
        expected[nan_rows], expected[:, nan_cols] = True, True
        assert np.array_equal(nan, expected), form
        assert np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32)), form


RING = (5, 6, 7, 8, 9)   # bench switch 15: the ring's tiles of 32 x 64, 64 x 64, 64 x 128, 128 x 64 and 128 x 128


@pytest.mark.parametrize("m,n,k", [(1, 1, 128), (17, 33, 192), (64, 32, 512), (65, 31, 576), (63, 66, 1984), (129, 130, 2048),
                                   (128, 128, 2112), (97, 257, 4160), (130, 127, 6656), (70, 65, 8128), (33, 129, 8192)])
def test_ring_is_bitwise_the_16_row_form(gpu, m, n, k):
    """Edges of every tile; k of one step, of a part of one, of steps that fill no four and no sixteen, and the longest."""
    a, a_s, w, w_s = md.gemm_case(m, n, k, 5)
    a_d, as_d, w_d, ws_d = dev(a), dev(a_s), dev(w), dev(w_s)
    shifted = dev(np.concatenate([np.zeros(1, np.uint8), w_s.reshape(-1)]))
    want = None
    for form in (1,) + RING:
        for scales, pad in ((ws_d, 4), (shifted[1:], 3)):
            out, outh = dev_empty((m, n + pad), np.float32), dev_empty((m, n + pad), np.uint16)
            out.fill_(-1)
            outh.fill_(0x55)
            before = _lib.load().dgpp_bench_tiled_launches()
            _lib.load().dgpp_tune_set(15, form)
            try:
                L.launch_mxfp8_gemm_f32(a_d, as_d, w_d, scales, out, m, n, k, None, n + pad)
                L.launch_mxfp8_gemm_bf16(a_d, as_d, w_d, scales, outh, m, n, k, None, n + pad)
            finally:
                _lib.load().dgpp_tune_set(15, 0)
            sync()
            if form < 9 or k <= 6656:   # the largest tile's panel is shorter
                assert _lib.load().dgpp_bench_tiled_launches() - before == (2 if form > 1 else 0)
            got = host(out).view(np.uint32)[:, :n].copy(), host(outh)[:, :n].copy()
            assert (host(out)[:, n:] == -1).all() and (host(outh)[:, n:] == 0x55).all()
            want = want or got
            for x, y in zip(want, got):
                assert np.array_equal(x, y), (form, m, n, k)


@pytest.mark.parametrize("k", [192, 2112])
def test_non_finite_codes_and_scales_in_the_ring(gpu, k):
    """Where k ends inside a step the ring reads the next row's bytes, here NaN codes, and clears them."""
    m, n = 70, 66
    a, a_s, w, w_s = md.gemm_case(m, n, k, 6)
    a[2, 0], a[30, k - 1], w[7, 0], w[65, k - 1] = 0x7F, 0xFF, 0x7F, 0xFF
    a_s[11, 0] = a_s[69, -1] = w_s[20, -1] = w_s[33, 1] = 0xFF
    nan_rows, nan_cols = [2, 11, 30, 69], [7, 20, 33, 65]
    ops = [dev(v) for v in (a, a_s, w, w_s)]
    out = dev_empty((m, n), np.float32)
    want = None
    for form in (1,) + RING:
        out.fill_(-1)
        _lib.load().dgpp_tune_set(15, form)
        try:
            L.launch_mxfp8_gemm_f32(*ops, out, m, n, k)
        finally:
            _lib.load().dgpp_tune_set(15, 0)
        sync()
        got = host(out).copy()
        want = got if want is None else want
        expected = np.zeros((m, n), bool)
        expected[nan_rows], expected[:, nan_cols] = True, True
        assert np.array_equal(np.isnan(got), expected), form
        assert np.array_equal(got[~expected].view(np.uint32), want[~expected].view(np.uint32)), form
