"""The matrix-core form for many activation rows (128 x 128 tiles) against the 16-row form, bit for bit: both add the
same products in the same order, and the 16-row form is held to the oracle in test_gpu_mma.py and test_gpu_w4a4.py.
Sizes at the edges of tiles: row tiles of 128 (gate + up: 64), passes of 32 / 64 / 128 activation rows, k tiles of 128
with remainders, one, two and four parts of k. Bench switch 15 pins the form: 1 the 16-row form, 2 the tiled one."""
import numpy as np
import pytest

import moe_data
from dgpp_amd import _lib, hostgen as hg, launch as L, moe_layer as ML
from gpu_util import DeviceMoe, dev, dev_empty, fp4_matrix, host, sync
from test_gpu_dense_gemv import make_fp4
from test_gpu_moe_layer import make_layer

pytestmark = pytest.mark.gpu


TILES = 2   # bench switch 15: the tiled form that both() compares, 2 of 128 activation rows, of dense products 5 of 64 and 6 of 32


def both(run, *outs, tiled=1):
    """The outputs of run() under the 16-row form and under the tiled one, in `tiled` launches of it (0: the rows are not
    aligned and the 16-row form stays)."""
    got = []
    for form in (1, TILES):
        for o in outs:
            o.fill_(-1 if o.dtype.is_floating_point else 0x55)
        _lib.load().dgpp_tune_set(15, form)
        before = _lib.load().dgpp_bench_tiled_launches()
        try:
            run()
        finally:
            _lib.load().dgpp_tune_set(15, 0)
        sync()
        assert _lib.load().dgpp_bench_tiled_launches() - before == (tiled if form == TILES else 0)
        got.append([host(o).copy() for o in outs])
    return got


def same(run, what, *outs, tiled=1):
    want, got = both(run, *outs, tiled=tiled)
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
        same(lambda: L.launch_mma_gemv_fp8e8m0_bf16(act_d, k, p_d, s_d, out, m, n, k, n + 4, 0, 5), kind, out, tiled=m > 1)
        return
    rs, cs = (7, 7) if kind == "fp8" else (5, 6)
    payload, _ = hg.encode_fp8_blocks(wf, 128, 128)
    scales = rng.uniform(0.5, 2.0, ((n + (1 << rs) - 1) >> rs, (k + (1 << cs) - 1) >> cs)).astype(np.float32) * 1e-3
    p_d, s_d = dev(payload), dev(scales)
    same(lambda: L.launch_mma_gemv_fp8_bf16(act_d, k, p_d, s_d, out, m, n, k, n + 4, rs, cs), kind, out, tiled=m > 1)   # a row keeps to the vector core


@pytest.mark.parametrize("kind", ["nvfp4", "mxfp4", "fp8", "fp8grid", "mxfp8"])
@pytest.mark.parametrize("m,n,k", [(17, 40, 576), (33, 130, 1152), (64, 128, 2304), (97, 257, 4096), (129, 300, 640)])
@pytest.mark.parametrize("form", [5, 6])
def test_dense_tiles_of_fewer_rows_are_bitwise_the_16_row_form(gpu, kind, m, n, k, form, monkeypatch):
    """Tiles of 64 and of 32 activation rows: their edges, one, two and four parts of k, k tiles whole and in part."""
    monkeypatch.setitem(globals(), "TILES", form)
    test_dense_tiled_is_bitwise_the_16_row_form(gpu, kind, m, n, k)


def fp8_bytes(n, k, seed):
    rng = np.random.default_rng(seed)
    return dev(rng.integers(0, 120, (n, k), dtype=np.uint8)), dev(rng.uniform(0.5, 2.0, ((n + 127) >> 7, (k + 127) >> 7)).astype(np.float32) * 1e-3)


@pytest.mark.parametrize("m,n,k,rows", [(949, 995, 384, 32), (1123, 850, 1024, 64), (1171, 1103, 960, 128)])
def test_the_rule_reaches_each_width_of_dense_tiles(gpu, m, n, k, rows):
    lib = _lib.load()
    assert lib.dgpp_bench_dense_tile_rows(0, 0, m, n, k, 0, 0) == rows
    p_d, s_d = fp8_bytes(n, k, m)
    act_d, got = dev(hg.normal_bf16(0xD00 + n, (m, k))), []
    for form in (0, 1):
        out = dev_empty((m, n), np.uint16)
        out.fill_(0x55)
        before = lib.dgpp_bench_tiled_launches()
        lib.dgpp_tune_set(15, form)
        try:
            L.launch_mma_gemv_fp8_bf16(act_d, k, p_d, s_d, out, m, n, k, n, 7, 7)
        finally:
            lib.dgpp_tune_set(15, 0)
        sync()
        assert lib.dgpp_bench_tiled_launches() - before == (form == 0)
        got.append(host(out).copy())
    assert np.array_equal(*got)


@pytest.mark.parametrize("m,n", [(5, 1000), (16, 4096), (8, 16390), (9, 16390)])
def test_rows_of_no_whole_vectors_take_the_other_forms_by_the_rule(gpu, m, n):
    """The parts of k side by side, in blocks of four and of two row groups, and row tiles: what the rule leaves to rows that do not
    stream. Same bits as the rows streamed."""
    lib, k = _lib.load(), 4096
    p_d, s_d = fp8_bytes(n, k, n)
    act, got = hg.normal_bf16(0xD10 + n, (m, k)), []
    wide = np.zeros((m, k + 1), np.uint16)
    wide[:, :k] = act
    lib.dgpp_tune_set(5, 2)
    try:
        for rows, stride in ((act, k), (wide, k + 1)):
            rows_d, out = dev(rows), dev_empty((m, n), np.float32)
            out.fill_(-7.0)
            before = lib.dgpp_bench_form_launches(2)
            L.launch_mma_gemv_fp8_f32(rows_d, stride, p_d, s_d, out, m, n, k, n, 7, 7)
            sync()
            assert lib.dgpp_bench_form_launches(2) - before == (stride == k)
            got.append(host(out).view(np.uint32).copy())
    finally:
        lib.dgpp_tune_set(5, 0)
    assert np.array_equal(*got)


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
    same(lambda: plain_f(odd, I + 2, segs, E, most, 0, d.views, 2, down, H, H, I, None, None, *more), "unaligned rows", down,
         tiled=0)
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


@pytest.mark.parametrize("kind,group", [("nvfp4", 16), ("mxfp4", 32)])
@pytest.mark.parametrize("m,n,k", [(129, 100, 1152), (300, 257, 2304), (64, 64, 576)])
def test_gate_and_up_apart_of_one_segment(gpu, kind, group, m, n, k):
    """The form that stores gate and up unmerged (the dense product by views), a lone segment spread over the XCDs."""
    k = {1152: 1024, 2304: 2048, 576: 640}[k] if kind == "nvfp4" else k
    p = moe_data.make_problem(2, k, 288, 1, 4, kind, 17 + m, shared_kind=None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    x = dev(hg.normal_bf16(0x9C0 + k, (m, k)))
    seg = dev(np.array([[0, m, 1]], np.int32))
    gate, up = dev_empty((m, n), np.uint16), dev_empty((m, n), np.uint16)
    same(lambda: L.launch_dense_mma_fp4_gate_up_bf16(x, k, seg, d.views, gate, up, m, n, k, None, group), kind, gate, up)
    same(lambda: L.launch_dense_mma_fp4_prod_bf16(x, k, seg, d.views, 1, up, m, n, k, None, group), "prod", up)


def w4a4_rows(x, rows, k):
    codes, gs = dev_empty((rows, k // 2), np.uint8), dev_empty((rows,), np.float32)
    scales = dev_empty((rows, _lib.load().dgpp_nvfp4_act_scale_stride(k)), np.uint8)
    L.launch_quantize_rows_nvfp4(x, k, rows, k, codes, scales, gs)
    return codes, scales, gs


@pytest.mark.parametrize("m,n,k", [(65, 130, 128), (129, 257, 1152), (300, 100, 4224), (33, 64, 2304)])
def test_dense_nvfp4_activations_tiled_is_bitwise_the_16_row_form(gpu, m, n, k):
    """k of one tile, of tiles that the parts do not divide, and of a last part that is empty (33 tiles, 12 to a part)."""
    act, payload, scales, glob = make_fp4(m, n, k, 0xA40 + k, 16)
    codes, a_s, gs = w4a4_rows(dev(act), m, k)
    p_d, s_d, g_d = dev(payload), dev(scales), dev(glob)
    out = dev_empty((m, n + 5), np.uint16)
    same(lambda: L.launch_dense_w4a4_bf16(codes, a_s, a_s.shape[1], gs, p_d, s_d, g_d, out, n + 5, m, n, k), "dense w4a4", out)


@pytest.mark.parametrize("H,I", [(192, 320), (64, 1088)])
def test_grouped_nvfp4_activations_tiled_with_a_part_of_a_k_tile(gpu, H, I):
    rows = [1, 0, 33, 130, 64, 17, 65, 32, 300]
    E, total = len(rows), sum(rows)
    p = moe_data.make_problem(E, H, I, 2, 8, "nvfp4", 71, shared_kind=None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    starts = np.concatenate([[0], np.cumsum(rows)[:-1]])
    segs = dev(np.array([[starts[i], rows[i], (i * 4) % E] for i in range(E)], np.int32))
    for which, n, k in ((0, I, H), (2, H, I)):
        codes, scales, gs = w4a4_rows(dev(hg.normal_bf16(0xB60 + k, (total, k))), total, k)
        out, outf = dev_empty((total, n + 4), np.uint16), dev_empty((total, n), np.float32)
        same(lambda: L.launch_moe_grouped_w4a4_bf16(codes, scales, gs, None, segs, E, 300, d.views, which, out, n + 4, n, k), "bf16", out)
        same(lambda: L.launch_moe_grouped_w4a4_f32(codes, scales, gs, None, segs, E, 300, d.views, which, outf, n, n, k), "f32", outf)


def same_with_nan(run, what, *outs):
    """As same(); a NaN stands for any NaN, and some of the values are."""
    want, got = both(run, *outs)
    for a, b in zip(want, got):
        v = [o if o.dtype == np.float32 else hg.bf16_to_f32(o.view(np.uint16)) for o in (a, b)]
        nan = np.isnan(v[0])
        assert nan.any() and not nan.all(), what
        assert np.array_equal(nan, np.isnan(v[1])) and np.array_equal(v[0][~nan], v[1][~nan]), what


@pytest.mark.parametrize("kind", ["nvfp4", "mxfp4", "fp8", "mxfp8", "w4a4"])
def test_non_finite_values_reach_the_same_outputs(gpu, kind):
    """Infinite and NaN activations in the first, an inner and the last element of a row, NaN scales and (FP8) codes of some
    weight rows, with a part of a k tile where the format has one."""
    m, n = 130, 140
    k = {"nvfp4": 1024, "mxfp4": 1152, "fp8": 1104, "mxfp8": 1120, "w4a4": 1152}[kind]
    rng = np.random.default_rng(5)
    act = hg.normal_bf16(0xC10, (m, k))
    if kind != "w4a4":
        act[3, 0], act[40, k - 1], act[77, k // 2], act[129, 0] = 0x7F80, 0x7FC0, 0xFF80, 0x7FC0
    act_d = dev(act)
    if kind in ("nvfp4", "mxfp4", "w4a4"):
        _, payload, scales, glob = make_fp4(1, n, k, 0xC20, 32 if kind == "mxfp4" else 16)
        scales[5, 0] = scales[139, -1] = 0xFF if kind == "mxfp4" else 0x7F
        p_d, s_d, g_d = dev(payload), dev(scales), dev(glob) if glob is not None else None
        if kind == "w4a4":
            codes, a_s, gs = w4a4_rows(act_d, m, k)
            a_s[9, 1] = 0x7F
            gs[64] = float("inf")
            out = dev_empty((m, n), np.uint16)
            same_with_nan(lambda: L.launch_dense_w4a4_bf16(codes, a_s, a_s.shape[1], gs, p_d, s_d, g_d, out, n, m, n, k), kind, out)
            return
        w = fp4_matrix(p_d, s_d, g_d, n, k, 32 if kind == "mxfp4" else 16)
        outf = dev_empty((m, n), np.float32)
        same_with_nan(lambda: L.launch_mma_gemv_fp4_f32(act_d, k, w, outf, m, n, k, n), kind, outf)
        return
    wf = hg.f32_to_bf16(hg.normal_f32(0xC30, (n, k), 0.02))
    out = dev_empty((m, n), np.uint16)
    if kind == "mxfp8":
        payload, scales = hg.encode_mxfp8(hg.bf16_to_f32(wf))
        payload[6, k - 1], payload[100, 0], scales[8, -1] = 0x7F, 0xFF, 0xFF
        p_d, s_d = dev(payload), dev(scales)
        same_with_nan(lambda: L.launch_mma_gemv_fp8e8m0_bf16(act_d, k, p_d, s_d, out, m, n, k, n, 0, 5), kind, out)
        return
    payload, _ = hg.encode_fp8_blocks(wf, 128, 128)
    payload[6, k - 1], payload[100, 0] = 0x7F, 0xFF
    scales = rng.uniform(0.5, 2.0, ((n + 127) >> 7, (k + 127) >> 7)).astype(np.float32) * 1e-3
    scales[1, -1] = np.inf
    p_d, s_d = dev(payload), dev(scales)
    same_with_nan(lambda: L.launch_mma_gemv_fp8_bf16(act_d, k, p_d, s_d, out, m, n, k, n, 7, 7), kind, out)


@pytest.mark.parametrize("kind,shared,launches", [("nvfp4", "nvfp4", 2), ("mxfp4", "mxfp4", 2), ("nvfp4", "fp8", 4), ("fp8", "fp8", 4),
                                                  ("fp8", None, 2)])
@pytest.mark.parametrize("E,T", [(17, 300), (6, 140)])
def test_a_layer_with_a_shared_expert_is_bitwise_its_16_row_form(gpu, kind, shared, launches, E, T):
    """A shared expert's segment, as long as the prompt, behind the routed ones or in launches of its own: its blocks go
    over all XCDs, a table of fewer segments than XCDs likewise."""
    p = moe_data.make_problem(E, 512, 256, 3, T, kind, 55 + E, shared_kind=shared, shared_I=256 if shared else None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    layer = make_layer(p, d, L.ROUTER_SOFTMAX_TOPK, 1.0, T)
    out = dev_empty((T, 512), np.uint16)
    same(lambda: layer.enqueue_prefill(d.x, 512, out, T), kind, out, tiled=launches)
    layer.close()


@pytest.mark.parametrize("T", [70, 200])
def test_a_layer_with_an_mxfp8_shared_expert_does_not_depend_on_its_projections_form(gpu, T):
    """The projections beside the routed chain, in the form that is faster alone and in the tiles (bench switch 17)."""
    p = moe_data.make_problem(24, 512, 256, 3, T, "nvfp4", 77, shared_kind=None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    mats = [hg.encode_mxfp8(hg.normal_f32(0xD00 + i, (n, k), 0.05)) for i, (n, k) in enumerate(((384, 512), (384, 512), (512, 384)))]
    pay, scales = [dev(m[0]) for m in mats], [dev(m[1]) for m in mats]
    cfg = L.make_config(512, 256, 24, 3, n_shared_experts=1, routed_scaling_factor=1.0, swiglu_limit=7.0, router_mode=L.ROUTER_SOFTMAX_TOPK)
    views = list((L.MoeExpertView * (d.views.numel() // 96)).from_buffer_copy(bytes(host(d.views))))
    layer = ML.MoeLayer(cfg, ML.EXPERTS_NVFP4, views, T, shared_inter=384, sh_payload=pay, sh_scales_e8m0=scales, router_gate=dev(p.router_gate))
    out, got = dev_empty((T, 512), np.uint16), []
    for form in (1, 2, 0):
        out.fill_(0x55)
        before = _lib.load().dgpp_bench_tiled_launches()
        _lib.load().dgpp_tune_set(17, form)
        try:
            layer.enqueue_prefill(d.x, 512, out, T)
        finally:
            _lib.load().dgpp_tune_set(17, 0)
        sync()
        tiled = _lib.load().dgpp_bench_tiled_launches() - before
        got.append((host(out).copy(), tiled))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][0], got[2][0])
    assert got[1][1] - got[0][1] == 3 and got[2][1] == got[1 if T == 200 else 0][1]
    layer.close()


@pytest.mark.parametrize("kind", ["fp8", "mxfp4", "nvfp4", "w4a4"])
@pytest.mark.parametrize("E,T,K", [(70, 301, 5), (300, 700, 3)])
def test_sorted_passes_of_a_skewed_table_are_bitwise_the_16_row_form(gpu, kind, E, T, K):
    """A table of passes enough to be sorted by width: an expert with all tokens, some with 33 to 128, with fewer and with
    none; more segments than a block has threads."""
    p = moe_data.make_problem(E, 512, 512, K, T, "nvfp4" if kind == "w4a4" else kind, 31 + E, shared_kind=None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    layer = make_layer(p, d, L.ROUTER_SOFTMAX_TOPK, 1.0, T)
    rng = np.random.default_rng(E)
    popular = 1.0 / np.arange(1, E - 9) ** 1.1      # the last ten have no rows
    ids = np.stack([np.concatenate([[0], 1 + rng.choice(E - 10, K - 1, replace=False, p=popular / popular.sum())]) for _ in range(T)])
    counts = np.bincount(ids.reshape(-1), minlength=E)
    assert counts[0] == T and (counts == 0).any() and ((counts > 64) & (counts <= 128)).any() and ((counts > 0) & (counts <= 32)).any()
    ids_d = dev(ids.astype(np.int32))
    w = dev(rng.uniform(0.1, 1.0, (T, K)).astype(np.float32))
    out = dev_empty((T, 512), np.uint16)
    if kind == "w4a4":
        same(lambda: layer.enqueue_prefill_routed_w4a4(d.x, 512, ids_d, w, out, T), kind, out, tiled=3)
    else:
        same(lambda: layer.enqueue_prefill_routed(d.x, 512, ids_d, w, out, T), kind, out, tiled=2)
    layer.close()


@pytest.mark.parametrize("kind", ["fp8", "mxfp4", "nvfp4", "w4a4"])
@pytest.mark.parametrize("E,T,K,H,I", [(70, 301, 5, 512, 512), (300, 700, 3, 512, 576), (12, 40, 3, 2048, 640), (5, 33, 1, 1152, 576), (64, 16, 8, 4096, 320)])
def test_narrow_passes_are_bitwise_the_16_row_form(gpu, kind, E, T, K, H, I):
    """The kernel of 32-row passes (bench switch 15: 3): dealt by segment and sorted, segments of no row, one, 16, 17, 32, 33 and
    of every token, one, two and four parts of k, k tiles whole and in part."""
    if kind in ("nvfp4", "w4a4") and H == 1152:
        H = 1536
    p = moe_data.make_problem(E, H, I, K, T, "nvfp4" if kind == "w4a4" else kind, 77 + E, shared_kind=None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    layer = make_layer(p, d, L.ROUTER_SOFTMAX_TOPK, 1.0, T)
    rng = np.random.default_rng(E)
    popular = 1.0 / np.arange(1, E) ** 1.1
    ids = np.stack([np.concatenate([[0], 1 + rng.choice(E - 1, K - 1, replace=False, p=popular / popular.sum())]) for _ in range(T)])
    ids_d, w = dev(ids.astype(np.int32)), dev(rng.uniform(0.1, 1.0, (T, K)).astype(np.float32))
    out, got = dev_empty((T, H), np.uint16), []
    for form in (1, 3):
        out.fill_(0x55)
        _lib.load().dgpp_tune_set(15, form)
        before = _lib.load().dgpp_bench_form_launches(1)
        try:
            if kind == "w4a4":
                layer.enqueue_prefill_routed_w4a4(d.x, H, ids_d, w, out, T)
            else:
                layer.enqueue_prefill_routed(d.x, H, ids_d, w, out, T)
        finally:
            _lib.load().dgpp_tune_set(15, 0)
        sync()
        assert _lib.load().dgpp_bench_form_launches(1) - before == (0 if form == 1 else 3 if kind == "w4a4" else 2)
        got.append(host(out, np.uint16).copy())
    layer.close()
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("kind", ["fp8", "mxfp4"])
def test_activation_rows_beyond_four_gigabytes(gpu, kind):
    """Rows that a buffer load does not reach, alone in a pass and beside near ones, and rows that end at its edge."""
    import torch
    H, I, E, T = 1152, 576, 2, 1_900_000
    if T * H * 2 * 1.1 > torch.cuda.mem_get_info()[0]:
        pytest.skip("not enough memory")
    p = moe_data.make_problem(E, H, I, 1, 4, kind, 5, shared_kind=None, limit=7.0, std=0.05)
    d = DeviceMoe(p)
    edge = (1 << 32) // (2 * H)
    rows = np.array([0, 1, edge - 2, edge - 1] + [edge, edge + 1, T - 1, 3], np.int32)
    x = torch.empty((T, H), dtype=torch.bfloat16, device=d.x.device)
    x[torch.from_numpy(rows).long().to(x.device)] = dev(hg.normal_bf16(0x99, (len(rows), H))).view(torch.bfloat16)
    segs = dev(np.array([[0, 3, 0], [3, 5, 1]], np.int32))
    act = dev_empty((len(rows), I), np.uint16)
    gu = L.launch_moe_grouped_mma_gate_up_swiglu if kind == "fp8" else L.launch_moe_grouped_mma_gate_up_swiglu_fp4
    more = () if kind == "fp8" else (d.fp4_group,)
    idx = dev(rows)
    same(lambda: gu(x, H, segs, E, 5, 0, d.views, act, I, I, H, 7.0, None, idx, *more), kind, act)


STREAM_SHAPES = [(1, 1, 4096), (8, 33, 5120), (9, 31, 2048), (16, 130, 1152), (17, 64, 2304), (33, 300, 512), (70, 257, 8192), (5, 40, 64),
                 (3, 96, 4224), (20, 70, 4160), (7, 33, 4576), (6, 50, 4352)]


@pytest.mark.parametrize("kind", ["nvfp4", "mxfp4", "fp8", "mxfp8"])
@pytest.mark.parametrize("m,n,k", STREAM_SHAPES)
def test_streaming_dense_form_is_bitwise_the_row_tile_form(gpu, kind, m, n, k):
    """The dense launch that streams its weights, a part of K to a wavefront, against the form that walks the parts in turn
    (bench switch 11: 4, 1): one to four parts, row groups and column tiles at their edges, tiles of k that are whole, part and
    none, rows that no vector load reads; FP4 at 4352, 4160 and 4576 has an empty part, the last two with a part tile before it."""
    if kind in ("nvfp4", "mxfp4"):
        group = 16 if kind == "nvfp4" else 32
        k = {"nvfp4": {1152: 1536, 2304: 640, 64: 512, 4224: 7168, 8192: 3072}, "mxfp4": {64: 576, 4224: 1152, 8192: 2304}}[kind].get(k, k)
        act, payload, scales, glob = make_fp4(m, n, k, 0xE10 + n + k, group)
        p_d, s_d = dev(payload), dev(scales)
        w = fp4_matrix(p_d, s_d, dev(glob) if glob is not None else None, n, k, group)
        run = lambda a, stride, out: L.launch_mma_gemv_fp4_f32(a, stride, w, out, m, n, k, n + 3)
    else:
        act = hg.normal_bf16(0xE11 + n, (m, k))
        wf = hg.normal_f32(0xE12 + n + k, (n, k), 0.02)
        if kind == "mxfp8":
            payload, scales = hg.encode_mxfp8(wf)
            fn, rs, cs = L.launch_mma_gemv_fp8e8m0_f32, 0, 5
        else:
            k_used = k - 16 if k > 64 else k
            act, wf, k = np.ascontiguousarray(act[:, :k_used]), np.ascontiguousarray(wf[:, :k_used]), k_used
            payload, _ = hg.encode_fp8_blocks(hg.f32_to_bf16(wf), 128, 128)
            scales = np.random.default_rng(n).uniform(0.5, 2.0, ((n + 127) >> 7, (k + 127) >> 7)).astype(np.float32) * 1e-3
            fn, rs, cs = L.launch_mma_gemv_fp8_f32, 7, 7
        p_d, s_d = dev(payload), dev(scales)
        run = lambda a, stride, out: fn(a, stride, p_d, s_d, out, m, n, k, n + 3, rs, cs)
    wide = np.zeros((m, k + 1), np.uint16)
    wide[:, :k] = act
    rows = [(dev(act), k), (dev(wide), k + 1)]
    lib, got = _lib.load(), []
    lib.dgpp_tune_set(5, 2)
    lib.dgpp_tune_set(15, 1)
    try:
        for knob in (1, 4):
            for a, stride in rows:
                before = lib.dgpp_bench_form_launches(2)
                lib.dgpp_tune_set(11, knob)
                out = dev_empty((m, n + 3), np.float32)
                out.fill_(-7.0)
                run(a, stride, out)
                sync()
                assert lib.dgpp_bench_form_launches(2) - before == (knob == 4 and stride == k), "streamed, if the rows are whole vectors"
                got.append(host(out).copy())
    finally:
        for key in (5, 11, 15):
            lib.dgpp_tune_set(key, 0)
    assert (got[0][:, :n] != -7.0).all() and (got[0][:, n:] == -7.0).all()
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint32), got[0].view(np.uint32))


@pytest.mark.parametrize("kind", ["nvfp4", "mxfp4", "fp8", "mxfp8"])
@pytest.mark.parametrize("tiles", [1, 2, 3, 5, 6, 7, 11, 66])
def test_walks_that_end_with_part_of_a_turn_are_bitwise_the_16_row_form(gpu, kind, tiles):
    """Whole tiles of k that are no whole turns of four: the walk's last steps, where less is on its way than its counted waits
    stand on. Every pass width, the 128-row passes and (grouped) the 32-row ones; 66 tiles in two (block FP8, MXFP8) or four parts."""
    k = tiles * (64 if kind in ("fp8", "mxfp8") else 128)
    n, rows = 140, [32, 64, 128, 5, 96]
    if kind == "mxfp8":
        payload, scales = hg.encode_mxfp8(hg.normal_f32(0xF10 + k, (n, k), 0.02))
        p_d, s_d = dev(payload), dev(scales)
        for m in rows[:3]:
            x, out = dev(hg.normal_bf16(0xF11 + m, (m, k))), dev_empty((m, n), np.uint16)
            same(lambda: L.launch_mma_gemv_fp8e8m0_bf16(x, k, p_d, s_d, out, m, n, k, n, 0, 5), f"{m} rows", out)
        return
    E, total = len(rows), sum(rows)
    d = DeviceMoe(moe_data.make_problem(E, k, 128, 2, 4, kind, 0xF20 + tiles, shared_kind=None, limit=7.0, std=0.05))
    x = dev(hg.normal_bf16(0xF21 + k, (total, k)))
    starts = np.concatenate([[0], np.cumsum(rows)[:-1]])
    segs = dev(np.array([[starts[i], rows[i], (i * 2) % E] for i in range(E)], np.int32))
    plain = L.launch_moe_grouped_mma_f32 if kind == "fp8" else L.launch_moe_grouped_mma_fp4_f32
    more = () if kind == "fp8" else (d.fp4_group,)
    out, got = dev_empty((total, 128), np.float32), []
    for form in (1, 2, 3):
        out.fill_(-7.0)
        _lib.load().dgpp_tune_set(15, form)
        before = [_lib.load().dgpp_bench_form_launches(f) for f in (0, 1)]
        try:
            plain(x, k, segs, E, max(rows), 0, d.views, 1, out, 128, 128, k, None, None, *more)
        finally:
            _lib.load().dgpp_tune_set(15, 0)
        sync()
        assert [_lib.load().dgpp_bench_form_launches(f) - b for f, b in zip((0, 1), before)] == [form == 2, form == 3]
        got.append(host(out).copy())
    assert (got[0] != -7.0).all()
    for g in got[1:]:
        assert np.array_equal(g.view(np.uint32), got[0].view(np.uint32))
