"""The matrix-core form for many activation rows (128 x 128 tiles) against the 16-row form, bit for bit: both add the
same products in the same order, and the 16-row form is held to the oracle in test_gpu_mma.py and test_gpu_w4a4.py.
Sizes at the edges of tiles: row tiles of 128 (gate + up: 64), passes of 32 / 64 / 128 activation rows, k tiles of 128
with remainders, one, two and four parts of k. Bench switch 15 pins the form: 1 the 16-row form, 2 the tiled one."""
import numpy as np
import pytest

import moe_data
from dgpp_amd import _lib, hostgen as hg, launch as L
from gpu_util import DeviceMoe, dev, dev_empty, fp4_matrix, host, sync
from test_gpu_dense_gemv import make_fp4

pytestmark = pytest.mark.gpu


def both(run, *outs):
    """The outputs of run() under the 16-row form and under the tiled one."""
    got = []
    for form in (1, 2):
        for o in outs:
            o.fill_(-1 if o.dtype.is_floating_point else 0x55)
        _lib.load().dgpp_tune_set(15, form)
        try:
            run()
        finally:
            _lib.load().dgpp_tune_set(15, 0)
        sync()
        got.append([host(o).copy() for o in outs])
    return got


def same(run, what, *outs):
    want, got = both(run, *outs)
    for a, b in zip(want, got):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), what


@pytest.mark.parametrize("kind", ["nvfp4", "mxfp4", "fp8", "fp8grid", "mxfp8"])
@pytest.mark.parametrize("m,n,k", [(1, 40, 576), (33, 130, 1152), (64, 128, 2304), (65, 257, 4096), (129, 1100, 640),
                                   (300, 100, 5120)])
def test_dense_tiled_is_bitwise_the_16_row_form(gpu, kind, m, n, k):
    if kind in ("nvfp4", "mxfp4"):
        group = 16 if kind == "nvfp4" else 32
        act, payload, scales, glob = make_fp4(m, n, k, 0x7A0 + n + k, group)
        act_d, p_d, s_d = dev(act), dev(payload), dev(scales)
        g_d = dev(glob) if glob is not None else None
        w = fp4_matrix(p_d, s_d, g_d, n, k, group)
        out, outf = dev_empty((m, n + 3), np.uint16), dev_empty((m, n + 4), np.float32)
        same(lambda: L.launch_mma_gemv_fp4_bf16(act_d, k, w, out, m, n, k, n + 3), f"bf16 {kind}", out)
        same(lambda: L.launch_mma_gemv_fp4_f32(act_d, k, w, outf, m, n, k, n + 4), f"f32 {kind}", outf)
        return
    if kind == "fp8grid":
        k -= 16 if m % 2 else 48       # an odd number of 16-element chunks; a part of a step
    rng = np.random.default_rng(n + k)
    wf = hg.f32_to_bf16(hg.normal_f32(0x8B0 + n + k, (n, k), 0.02))
    act_d = dev(hg.normal_bf16(0x8B1 + n, (m, k)))
    out = dev_empty((m, n + 4), np.uint16)
    if kind == "mxfp8":
        payload, scales = hg.encode_mxfp8(hg.bf16_to_f32(wf))
        p_d, s_d = dev(payload), dev(scales)
        same(lambda: L.launch_mma_gemv_fp8e8m0_bf16(act_d, k, p_d, s_d, out, m, n, k, n + 4, 0, 5), kind, out)
        return
    rs, cs = (7, 7) if kind == "fp8" else (5, 6)
    payload, _ = hg.encode_fp8_blocks(wf, 128, 128)
    scales = rng.uniform(0.5, 2.0, ((n + (1 << rs) - 1) >> rs, (k + (1 << cs) - 1) >> cs)).astype(np.float32) * 1e-3
    p_d, s_d = dev(payload), dev(scales)
    same(lambda: L.launch_mma_gemv_fp8_bf16(act_d, k, p_d, s_d, out, m, n, k, n + 4, rs, cs), kind, out)


@pytest.mark.parametrize("kind", ["nvfp4", "mxfp4", "fp8"])
@pytest.mark.parametrize("H,I", [(1152, 576), (2048, 640)])
def test_grouped_tiled_is_bitwise_the_16_row_form(gpu, kind, H, I):
    """Segments of every pass width and none at all, more than one pass long, gathered and in place; the z rule's passes
    in turn (bench switch 16 = 1) and side by side."""
    if kind == "nvfp4":
        H, I = {1152: 1024, 2048: 2048}[H], {576: 640, 640: 768}[I]
    if kind == "mxfp4" and I == 640:
        I = 1024
    rows = [1, 0, 33, 130, 64, 301, 17, 128, 65, 32]
    E, total, T = len(rows), sum(rows), 90
    p = moe_data.make_problem(E, H, I, 2, T, kind, 91, shared_kind=None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    rng = np.random.default_rng(H)
    starts = np.concatenate([[0], np.cumsum(rows)[:-1]])
    segs = dev(np.array([[starts[i], rows[i], (i * 7) % E] for i in range(E)], np.int32))
    idx = dev(rng.integers(0, T, total).astype(np.int32))
    most = max(rows)
    act, gate, up = (dev_empty((total, I + 4), np.uint16) for _ in range(3))
    down, down_odd = dev_empty((total, H), np.float32), dev_empty((total, H + 1), np.float32)
    slot = dev(hg.normal_bf16(0x77, (total, I)))
    more = () if kind == "fp8" else (d.fp4_group,)
    gu = L.launch_moe_grouped_mma_gate_up_swiglu if kind == "fp8" else L.launch_moe_grouped_mma_gate_up_swiglu_fp4
    plain = L.launch_moe_grouped_mma_bf16 if kind == "fp8" else L.launch_moe_grouped_mma_fp4_bf16
    plain_f = L.launch_moe_grouped_mma_f32 if kind == "fp8" else L.launch_moe_grouped_mma_fp4_f32
    for passes in (0, 1):
        _lib.load().dgpp_tune_set(16, passes)
        try:
            same(lambda: gu(d.x, H, segs, E, most, 0, d.views, act, I + 4, I, H, 7.0, None, idx, *more), "gate+up", act)
            same(lambda: plain(d.x, H, segs, E, most, 0, d.views, 1, up, I + 4, I, H, None, idx, *more), "up", up)
            same(lambda: plain_f(slot, I, segs, E, most, 0, d.views, 2, down, H, H, I, None, None, *more), "down", down)
        finally:
            _lib.load().dgpp_tune_set(16, 0)
    same(lambda: plain_f(slot, I, segs, E, most, 0, d.views, 2, down_odd, H + 1, H, I, None, None, *more), "odd stride", down_odd)
    # rows that are no whole 16-byte vectors keep the 16-row form
    odd = dev(hg.normal_bf16(0x79, (total, I + 2)))
    same(lambda: plain_f(odd, I + 2, segs, E, most, 0, d.views, 2, down, H, H, I, None, None, *more), "unaligned rows", down)
    if kind == "nvfp4":
        codes, gs = dev_empty((T, H // 2), np.uint8), dev_empty((T,), np.float32)
        scales = dev_empty((T, _lib.load().dgpp_nvfp4_act_scale_stride(H)), np.uint8)
        L.launch_quantize_rows_nvfp4(d.x, H, T, H, codes, scales, gs)
        same(lambda: L.launch_moe_grouped_w4a4_bf16(codes, scales, gs, idx, segs, E, most, d.views, 0, gate, I + 4, I, H),
             "w4a4 gate", gate)
        c2, g2 = dev_empty((total, I // 2), np.uint8), dev_empty((total,), np.float32)
        s2 = dev_empty((total, _lib.load().dgpp_nvfp4_act_scale_stride(I)), np.uint8)
        L.launch_quantize_rows_nvfp4(slot, I, total, I, c2, s2, g2)
        same(lambda: L.launch_moe_grouped_w4a4_f32(c2, s2, g2, None, segs, E, most, d.views, 2, down, H, H, I), "w4a4 down", down)
