"""The tile for a dense 32-packed layer, by prices, with the filter in the reference layout and pre-processed: near the best of the tiles timed,
and the result of the generic kernel over odd sizes, strides, gaps between images, residuals and destination types."""
import numpy as np
import pytest

from megengine_amd import _abi, lib, ops

S = dict(scale_bias=2e-4, scale_z=0.05, scale_dst=0.05)
# n, ic, h, w, oc, f, stride, residual, pre-processed; tiles within 6 % of the best in graph replays on 256 CUs, best first
LAYERS = [
    (2, 32, 54, 24, 32, 3, 1, 1, 0, "v2_ks_32x32w4 v2_ks_16x16w4 v2_patch_32x128"),
    (45, 192, 34, 9, 32, 1, 2, 1, 0, "v2_ks_32x32w4 v2_ks_16x16w4 v2_ks_16x16w8"),
    (29, 96, 10, 52, 32, 3, 2, 1, 0, "v2_ks_32x32w4 v2_ks_16x16w4"),
    (1, 384, 12, 21, 320, 1, 1, 1, 0, "v2_ks_32x32w4 v2_ks_16x16w4"),
    (9, 64, 26, 11, 1568, 1, 2, 1, 0, "dma64x64x64r4"),
    (37, 192, 70, 23, 160, 3, 2, 0, 0, "dma64x64x128r2 dma128x128x64w8 dma128x128x128r2w8 v2_128x128x64r4w8 dma64x128x128w8"),
    (4, 64, 13, 24, 480, 1, 2, 0, 0, "v2_ks_32x32w4 pw32_stream v2_ks_32x32w8 dma64x64x64r4"),
    (9, 128, 41, 95, 128, 3, 1, 0, 0, "dma128x128x128r2w8 v2_128x256x64r3w8"),
    (18, 256, 8, 48, 736, 5, 2, 0, 0, "dma64x128x128w8 dma64x64x128"),
    (27, 160, 37, 24, 128, 1, 1, 0, 0, "v2_128x128x64r4 v2_64x128x64r4 v2_64x128x64r5 v2_64x128x128r3 v2_128x64x64r4 v2_128x128x64r4w8"),
    (1, 608, 101, 27, 96, 3, 2, 0, 0, "v2_ks_16x16w4 v2_ks_16x16w8"),
    (16, 224, 41, 82, 64, 1, 1, 0, 0, "v2_64x128x64r4 v2_64x128x128r3 dma128x128x128r2w8 dma64x64x128r2 v2_64x128x64r5 v2_64x64x128r3"),
    (2, 640, 7, 35, 448, 3, 2, 1, 0, "v2_ks_16x16w4 v2_ks_16x16w8"),
    (3, 224, 19, 10, 384, 1, 1, 0, 0, "v2_ks_32x32w4 v2_ks_64x32w8 v2_64x64x128r4 v2_ks_64x32w4"),
    (12, 96, 101, 72, 384, 3, 1, 0, 0, "v2_128x256x64r3w8"),
    (42, 640, 18, 22, 1056, 3, 2, 0, 0, "dma128x128x128r2w8"),
    (23, 64, 9, 7, 32, 1, 1, 0, 1, "pw32_stream v2_ks_16x16w4"),
    (26, 128, 7, 7, 32, 5, 2, 1, 1, "v2_ks_16x16w8"),
    (28, 672, 42, 9, 32, 1, 1, 1, 1, "v2_ks_32x32w4"),
    (28, 512, 5, 5, 2048, 1, 1, 1, 1, "dma64x64x128 dma64x128x128w8 dma64x64x64r4 v2_ks_64x32w4 dma64x64x128r2"),
    (4, 512, 24, 24, 256, 1, 1, 0, 1, "v2_64x64x128r3 v2_64x64x128r4 dma64x64x128 dma64x64x128r2 v2_ks_64x32w4 dma64x64x64r4"),
    (24, 512, 32, 32, 1024, 1, 2, 0, 1, "dma128x128x128r2w8 dma128x64x128r2 v2_128x128x64r4 dma128x64x128w8 v2_128x64x64r4 v2_128x128x64r4w8"),
    (2, 64, 10, 10, 864, 3, 1, 0, 1, "v2_ks_32x32w4"),
    (4, 160, 29, 20, 160, 3, 2, 1, 1, "v2_ks_32x32w8 v2_ks_32x32w4 v2_ks_16x16w4"),
    (1, 512, 5, 5, 512, 3, 1, 0, 1, "v2_ks_16x16w8"),
    (26, 512, 4, 4, 2048, 1, 1, 1, 1, "v2_ks_64x32w4 v2_ks_64x32w8 v2_ks_32x32w4"),
    (8, 512, 6, 6, 2048, 1, 1, 1, 1, "v2_ks_32x32w4 v2_ks_64x32w4 v2_ks_64x32w8"),
    (4, 448, 49, 23, 1888, 3, 1, 0, 1, "v2_128x128x64r3 v2_128x128x64r4"),
    (38, 736, 64, 7, 64, 3, 1, 1, 1, "v2_64x64x128r4 dma64x128x128w8 v2_64x64x128r3"),
    (61, 128, 30, 30, 512, 1, 1, 1, 1, "pw32_stream dma128x128x128r2w8 dma128x128x64w8 128x128x64"),
    (20, 128, 31, 41, 160, 1, 1, 1, 1, "dma64x64x128r2 dma64x64x128 dma64x64x64r4"),
    (5, 64, 32, 32, 64, 3, 1, 0, 1, "v2_patch_32x128 v2_ks_32x32w4"),
]


def test_near_the_best():
    names, miss = lib.tile_names(), []
    for n, ic, h, w, oc, f, s, z, pre, near in LAYERS:
        d = _abi.make_conv_desc("NCHW32", n, ic, h, w, oc, f, pad=f // 2, stride=s, nonline="RELU", has_z=bool(z), **S)
        a, _ = ops.conv_bias_query(d, _abi.ALGO_HEURISTIC_PREPROCESS if pre else _abi.ALGO_HEURISTIC)
        assert a.id == 1 and lib.tile_usable(d, a.tile_cfg)
        if names[a.tile_cfg] not in near.split():
            miss.append((n, ic, h, w, oc, f, s, z, pre, names[a.tile_cfg], near))
    # over 26000 other layers the pick is 3.4 % behind the best on average, more than 10 % on 13 in a hundred
    assert len(miss) <= len(LAYERS) // 6, miss


def _draw(rng):
    lg = lambda lo, hi: int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))
    f = int(rng.choice([1, 1, 3, 5]))
    fmt = str(rng.choice(["NCHW32", "NCHW32", "NCHW32", "NCHW32_NCHW4"]))
    n, ic, h, w, oc, s = lg(1, 64), 32 * lg(1, 20), lg(2, 60), lg(2, 60), 32 * lg(1, 16), int(rng.choice([1, 1, 2]))
    n = max(1, min(n, int(1e10 / (h * w * oc * ic * f * f))))
    kw = dict(nonline=str(rng.choice(["IDENTITY", "RELU", "H_SWISH"])))
    if fmt == "NCHW32" and rng.randint(5) == 0:
        d = _abi.make_conv_desc(fmt, n, ic, h, w, oc, f, pad=f // 2, stride=s, dst_dtype=_abi.DT_QS32, scale_bias=2e-4, scale_dst=2e-4, **kw)
    else:
        d = _abi.make_conv_desc(fmt, n, ic, h, w, oc, f, pad=f // 2, stride=s, has_z=fmt == "NCHW32" and rng.randint(3) == 0, **S, **kw)
    if rng.randint(4) == 0:
        d.src_stride_n = ic * h * w + 32 * int(rng.randint(1, 9))
    return d


@pytest.mark.gpu
def test_against_the_generic_kernel():
    import torch
    rng = np.random.RandomState(17)
    used = set()
    for it in range(60):
        d = _draw(rng)
        ss, fs, bs, ds = _abi.conv_shapes(d)
        g = torch.Generator().manual_seed(it)
        s8 = lambda shape: torch.randint(-128, 128, shape, generator=g, dtype=torch.int8).cuda()
        src = s8((d.n, d.src_stride_n) if d.src_stride_n else ss)
        flt, z = s8(fs), s8(ds) if d.has_z else None
        bias = torch.randint(-4000, 4000, bs, generator=g, dtype=torch.int32).cuda()
        dt = torch.int32 if d.dst_dtype == _abi.DT_QS32 else torch.int8
        direct, _ = ops.conv_bias_query(d, 0)
        want = ops.conv_bias_exec(d, src, flt, bias, z, torch.empty(ds, dtype=dt, device="cuda"), direct)
        for req in (_abi.ALGO_HEURISTIC, _abi.ALGO_HEURISTIC_PREPROCESS):
            a, ws = ops.conv_bias_query(d, req)
            print("case", it, list(d.key())[:20], lib.tile_names()[a.tile_cfg], flush=True)
            out = torch.empty(ds, dtype=dt, device="cuda")
            pre = ops.conv_bias_preprocess(d, flt, a) if req == _abi.ALGO_HEURISTIC_PREPROCESS else None
            if pre is None:
                ops.conv_bias_exec(d, src, flt, bias, z, out, a)
            else:
                ops.conv_bias_exec_preprocessed(d, src, pre, bias, z, out, a)
            used.add(lib.tile_names()[a.tile_cfg])
            assert torch.equal(out, want), (it, list(d.key()), lib.tile_names()[a.tile_cfg])
    assert len(used) >= 8, used


# n, ic, h, w, oc, f, stride, residual, pre-processed; us (graph replays on 256 CUs) on the tile that the busiest XCD has least of, and on
# the one that fewer tiles in all spoke for
BUSIEST_XCD = [
    (3, 416, 10, 22, 576, 3, 1, 0, 0, "v2_ks_32x32w4", 9.2, "v2_ks_64x32w8", 16.7),
    (5, 512, 25, 9, 160, 3, 2, 1, 0, "v2_ks_16x16w4", 6.2, "v2_ks_16x16w8", 8.9),
    (10, 448, 12, 17, 576, 3, 2, 0, 0, "v2_ks_32x32w8", 11.9, "v2_ks_64x32w8", 16.6),
    (2, 256, 10, 78, 160, 5, 1, 0, 0, "v2_ks_64x32w8", 11.5, "v2_ks_32x32w8", 15.2),
    (4, 864, 11, 18, 160, 5, 1, 1, 1, "v2_ks_32x32w8", 15.8, "v2_ks_16x16w8", 24.3),
    (9, 288, 13, 22, 288, 5, 2, 0, 1, "v2_ks_64x32w8", 9.5, "v2_ks_32x32w8", 13.2),
    (4, 352, 16, 10, 288, 3, 1, 0, 1, "v2_ks_64x32w8", 5.2, "v2_ks_32x32w4", 6.7),
    (3, 416, 42, 20, 608, 5, 2, 0, 1, "v2_ks_32x32w4", 17.5, "v2_ks_64x32w8", 22.0),
]


def test_tiles_are_counted_by_the_busiest_xcd():
    names = lib.tile_names()
    for n, ic, h, w, oc, f, s, z, pre, best, us, other, other_us in BUSIEST_XCD:
        d = _abi.make_conv_desc("NCHW32", n, ic, h, w, oc, f, pad=f // 2, stride=s, nonline="RELU", has_z=bool(z), **S)
        a, _ = ops.conv_bias_query(d, _abi.ALGO_HEURISTIC_PREPROCESS if pre else _abi.ALGO_HEURISTIC)
        assert us < 0.8 * other_us and names[a.tile_cfg] == best, (n, ic, oc, names[a.tile_cfg])
