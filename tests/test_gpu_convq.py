"""GPU parity tests of the Conv2d_q forward (C ABI): int32 accumulators and requantized uint8 outputs bit-exact against
the oracle, the golden outputs of l-ten's compiled Conv2d_q layer, and the int64 closed form."""
import numpy as np
import pytest

from conftest import golden_path
from test_oracle_conv import conv2dq_closed_form

pytestmark = pytest.mark.gpu


def test_conv2dq_golden_from_compiled_layer(gpu):
    g = np.load(golden_path("conv2dq_cases.npz"))
    for variant in (0, 1):   # 0: the library's choice (one launch up to 64 taps); 1: im2col + GEMM per image
        gpu.set_option("conv_variant", variant)
        try:
            for i in range(int(g["count"])):
                pre = f"q{i}_"
                geo = tuple(int(v) for v in g[pre + "geo"])
                y, acc = gpu.conv2dq_host(geo, g[pre + "x"], g[pre + "w"], g[pre + "scales"], g[pre + "zps"], want_acc=True)
                assert np.array_equal(y, g[pre + "y"]), (variant, i, gpu.last_kernel())
                want = conv2dq_closed_form(geo, g[pre + "x"], g[pre + "w"], int(g[pre + "zps"][0]), int(g[pre + "zps"][1]))
                assert np.array_equal(acc, want), (variant, i)
        finally:
            gpu.set_option("conv_variant", 0)


@pytest.mark.parametrize("geo", [(64, 1, 28, 28, 10, 5, 5, 0, 0, 1, 1),      # l-ten's quantized MNIST conv1 at batch 64
                                 (3, 7, 13, 17, 70, 3, 3, 1, 1, 1, 1),       # 63 taps, two channel blocks
                                 (2, 16, 20, 22, 24, 3, 3, 1, 1, 2, 1),      # 144 taps: patch rows + GEMM + finish
                                 (5, 10, 12, 12, 20, 5, 5, 0, 0, 1, 1),      # l-ten's quantized MNIST conv2: 250 taps (padded to 256)
                                 (3, 8, 9, 7, 10, 3, 3, 1, 1, 1, 1),         # 72 taps, 63 positions an image
                                 (3, 15, 9, 7, 10, 3, 3, 1, 1, 1, 1),        # 135 taps, 10 channels (padded to 12), 63 positions an image
                                 (2, 64, 6, 10, 70, 3, 3, 1, 1, 1, 1),       # 576 taps, two channel blocks of the finish pass
                                 (4, 128, 5, 5, 33, 1, 1, 0, 0, 1, 1),       # 1x1 with 128 channels
                                 (2, 6, 14, 14, 16, 5, 5, 2, 2, 1, 1),       # 150 taps, padding 2
                                 (1, 20, 17, 9, 6, 3, 5, 0, 2, 2, 2),        # 300 taps, strides, oblong window
                                 (1, 3, 33, 300, 5, 7, 3, 3, 0, 2, 3),       # 63 taps, strides, ragged
                                 (2, 32, 9, 9, 40, 1, 1, 0, 0, 1, 1),        # 1x1
                                 (2, 5, 11, 13, 9, 3, 3, 1, 0, 1, 2),        # 45 taps: twelve packed dwords
                                 (1, 4, 8, 8, 3, 2, 2, 1, 1, 1, 1),          # 16 taps: four dwords, all full
                                 (2, 11, 7, 9, 5, 1, 3, 0, 1, 1, 1),         # 33 taps: one tap in the ninth dword
                                 (1, 3, 12, 10, 7, 4, 4, 1, 2, 1, 1),        # 48 taps
                                 (64, 10, 12, 12, 20, 5, 5, 0, 0, 1, 1),     # l-ten's quantized MNIST conv2 at batch 64
                                 (3, 9, 15, 11, 64, 3, 3, 1, 1, 1, 1),       # 81 taps, four blocks of 16 channels, 165 positions
                                 (2, 16, 28, 32, 17, 3, 3, 2, 2, 1, 1),      # 144 taps, 1020 positions an image: 64 workgroups each
                                 (2, 40, 5, 5, 30, 5, 5, 2, 2, 1, 1),        # 1000 taps, most of them outside the image
                                 (2, 40, 5, 5, 50, 5, 5, 2, 2, 1, 1),        # the same with 50 channels: weights beyond the 64 KB of LDS the route allows
                                 (1, 33, 31, 31, 3, 2, 2, 0, 0, 3, 3),       # 132 taps, image of 31.7 KB, stride 3
                                 (1, 65, 9, 9, 70, 1, 1, 0, 0, 1, 1),        # 65 taps but 70 channels: not for the one-launch route
                                 (2, 16, 40, 40, 24, 3, 3, 1, 1, 1, 1),      # 1600 positions an image: bands of output rows
                                 (1, 8, 50, 70, 64, 5, 3, 2, 1, 2, 1),       # bands with a row stride of 2, 64 channels, 120 taps
                                 (1, 3, 100, 37, 9, 5, 5, 0, 0, 1, 1),       # rows of 37 bytes: the region is filled byte by byte
                                 (3, 12, 33, 41, 20, 3, 3, 0, 2, 1, 3),      # column stride 3, padding 2 on the columns only
                                 (1, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1),      # 576 taps, 64 channels: several passes of blocks per band
                                 (3, 8, 44, 36, 16, 5, 5, 2, 2, 1, 1),       # bands, 5 x 5 windows of 8 channels (weights permuted in registers, 25 taps)
                                 (2, 4, 67, 70, 12, 7, 7, 3, 3, 2, 2),       # bands, 7 x 7 windows of 4 channels, stride 2 (49 taps)
                                 (19, 12, 36, 36, 40, 3, 3, 1, 1, 1, 1),     # 19 images x 9 bands = 171 workgroups: not a multiple of the 8 XCDs
                                 (2, 16, 20, 24, 80, 3, 3, 1, 1, 1, 1),      # 80 channels: a block of 64 and one of 16 per band
                                 (1, 128, 14, 14, 136, 3, 3, 1, 1, 1, 1),    # 1152 taps: weights of 32 channels at a time fit LDS, 5 blocks
                                 (1, 400, 9, 9, 40, 3, 3, 0, 0, 1, 1),       # 3600 taps: the weights of 32 channels do not fit, three launches
                                 (1, 200, 9, 9, 30, 3, 3, 0, 0, 1, 1),       # 1800 taps, 30 channels: two blocks of 16 channels
                                 (3, 96, 20, 20, 72, 1, 1, 0, 0, 1, 1),      # a 1 x 1 layer of 96 channels: the weights are copied as they lie
                                 (2, 68, 21, 22, 40, 1, 1, 1, 0, 2, 1),      # 1 x 1 with a row stride of 2 and padded rows
                                 (8, 16, 20, 24, 64, 2, 2, 0, 0, 2, 2),      # 64 taps, 64 channels: short windows on the band kernel
                                 (2, 3, 40, 44, 64, 3, 3, 1, 1, 1, 1),       # 27 taps of 3 channels (padded to 4), one k-step
                                 (2, 64, 12, 12, 80, 1, 1, 0, 0, 1, 1),      # 1 x 1 with 64 channels in, 80 out
                                 (3, 5, 17, 19, 50, 3, 3, 2, 2, 1, 2)])      # 45 taps, 50 channels, ragged everything
def test_conv2dq_vs_oracle(gpu, ob, geo):
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo))
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    Ho, Wo = ob.conv_out_hw(H, W, kh, kw, ph, pw, sh, sw)
    K = Cin * kh * kw
    for sc, zp, with_bias in (([1 / 255, 0.01, 0.05], [0, 128, 128], False), ([0.02, 0.013, 0.9], [17, 250, 100], True),
                              ([0.5, 0.5, 0.2], [128, 128, 0], False)):
        bias = rng.integers(-9999, 9999, Ho * Wo).astype(np.int32) if with_bias else None
        want_y, want_acc = ob.conv2dq_forward(geo, x, w, sc, zp, bias=bias)
        y, acc = gpu.conv2dq_host(geo, x, w, sc, zp, bias=bias, want_acc=True)
        kern = gpu.last_kernel()
        # up to 64 taps: one launch from registers; longer windows on small images: one launch from the image in LDS;
        # else patch rows + GEMM + finish
        Kp, ncb = (K + 63) // 64 * 64, (Cout + 15) // 16
        lds = (Cin * H * W + 15) // 16 * 16 + ncb * 16 * (Kp + 16) + 4 * Kp
        small = (Cin * H * W <= 32768 and Cout <= 64 and K <= 1024 and Ho * Wo <= 1024 and lds <= 65536 and
                 N * ((Ho * Wo + 15) // 16) <= 4096)
        # larger images with at most 64 channels: a band of output rows per workgroup, as long as one row's region fits LDS
        PL = (pw + 3) // 4 * 4
        RW = (PL + max((Wo - 1) * sw + kw - pw, W) + 3) // 4 * 4
        CP = 4 if Cin <= 4 else 8 if Cin <= 8 else 16
        CPtot = (Cin + CP - 1) // CP * CP
        PP = CPtot + (16 if CPtot % 32 == 0 else 0)
        Kb = (kh * kw * CPtot + 63) // 64 * 64      # the band kernel reduces over (tap, channel padded to a multiple of CP)
        # (blocks of 64 output channels per workgroup, or 32 where the weights of 64 leave no room for one window's rows; 16
        # only for layers of at most 32 channels)
        band = (pw <= 64 and kh * kw * CPtot <= 4096 and
                kh * RW * PP + (1 if ncb <= 2 else 2) * 16 * (Kb + 16) + 4 * (Kb // CP) + 2 * K + 32 <= 65536)
        # (where the band kernel applies, the small-image kernel only while its workgroups stage at most 16 MB in all and
        # the window is none of those whose weights the band kernel permutes in registers)
        staged = N * ((Ho * Wo + 15) // 16) * ((Cin * H * W + 15) // 16 * 16 + ncb * 16 * Kp)
        permuted = Cin % 4 == 0 and kh * kw in (1, 9, 25, 49)
        small = small and not (band and (permuted or staged > 16 << 20))
        # (windows of at most 64 taps: the band kernel from 48 output channels on, else one launch from registers)
        assert kern == (("conv2dq_band" if Cout >= 48 and band else "conv2dq_direct") if K <= 64 else
                        "conv2dq_image" if small else "conv2dq_band" if band else "conv2dq_rows_gemm_finish"), kern
        assert np.array_equal(acc, want_acc), kern
        assert np.array_equal(y, want_y), kern
        if kern in ("conv2dq_image", "conv2dq_band"):   # the three-launch route on the same shape gives the same bytes
            gpu.set_option("conv_variant", 2)
            try:
                y2, acc2 = gpu.conv2dq_host(geo, x, w, sc, zp, bias=bias, want_acc=True)
                assert gpu.last_kernel() == ("conv2dq_direct" if K <= 64 else "conv2dq_rows_gemm_finish")
            finally:
                gpu.set_option("conv_variant", 0)
            assert np.array_equal(acc2, want_acc) and np.array_equal(y2, want_y)
        if kern == "conv2dq_image" and band:   # and so does the band kernel where both one-launch kernels apply
            gpu.set_option("conv_variant", 3)
            try:
                y3, acc3 = gpu.conv2dq_host(geo, x, w, sc, zp, bias=bias, want_acc=True)
                assert gpu.last_kernel() == "conv2dq_band"
            finally:
                gpu.set_option("conv_variant", 0)
            assert np.array_equal(acc3, want_acc) and np.array_equal(y3, want_y)
    if K > 64:   # l-ten's decomposition image by image (what a workspace beyond 2 GiB falls back to) gives the same bytes
        gpu.set_option("conv_variant", 1)
        try:
            y1, acc1 = gpu.conv2dq_host(geo, x, w, sc, zp, bias=bias, want_acc=True)
            assert gpu.last_kernel() != "conv2dq_rows_gemm_finish"
        finally:
            gpu.set_option("conv_variant", 0)
        assert np.array_equal(acc1, want_acc) and np.array_equal(y1, want_y)


def test_conv2dq_long_windows_on_small_maps_take_the_three_launches(gpu, ob):
    """A 1 x 1 layer of 1024 channels on 14 x 14 maps: the band kernel has a plan (one output row and 32 channels per
    workgroup), but its workgroups would stage more than they compute, and the library's estimate sends the layer to patch
    rows + GEMM + finish.  Both routes give the oracle's bytes."""
    geo = (16, 1024, 14, 14, 256, 1, 1, 0, 0, 1, 1)
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo))
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    sc, zp = [0.02, 0.013, 0.9], [17, 250, 100]
    want_y, want_acc = ob.conv2dq_forward(geo, x, w, sc, zp)
    y, acc = gpu.conv2dq_host(geo, x, w, sc, zp, want_acc=True)
    assert gpu.last_kernel() == "conv2dq_rows_gemm_finish", gpu.last_kernel()
    assert np.array_equal(acc, want_acc) and np.array_equal(y, want_y)
    gpu.set_option("conv_variant", 3)   # the band kernel whatever the estimate says
    try:
        y3, acc3 = gpu.conv2dq_host(geo, x, w, sc, zp, want_acc=True)
        assert gpu.last_kernel() == "conv2dq_band", gpu.last_kernel()
    finally:
        gpu.set_option("conv_variant", 0)
    assert np.array_equal(acc3, want_acc) and np.array_equal(y3, want_y)


def conv2dq_at(gpu, geo, x, w, sc, zp, bias, off):
    """conv2dq_forward with every tensor `off` bytes past its buffer's start (the bias 4 off); the output between guard bytes."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    D = gpu.DeviceBuffer
    put = lambda a, o: D.from_numpy(np.concatenate([np.zeros(o, np.uint8), a.reshape(-1).view(np.uint8)]))
    dx, dw = put(x, off), put(w, off)
    db = put(bias, 4 * off) if bias is not None else None
    count = N * Cout * ((H + 2 * ph - kh) // sh + 1) * ((W + 2 * pw - kw) // sw + 1)
    ws_bytes = int(gpu.lib().lten_hip_conv2dq_workspace_bytes(*geo))
    ws, dy = D(ws_bytes + 64), D(count + off + 32)
    gpu.check(gpu.lib().lten_hip_fill_u8(dy.ptr, count + off + 32, 0xA5))
    gpu.check(gpu.lib().lten_hip_fill_u8(ws.ptr, ws_bytes + 64, 0x5A))
    gpu.check(gpu.lib().lten_hip_conv2dq_forward(*geo, dx.ptr + off, dw.ptr + off, db.ptr + 4 * off if db else None, gpu.qparams3(sc, zp),
                                                 dy.ptr + off, ws.ptr))
    got = dy.numpy(np.uint8, (count + off + 32,))
    assert (got[:off] == 0xA5).all() and (got[off + count:] == 0xA5).all(), "bytes beside the output were written"
    left = 0 if gpu.last_kernel() == "conv2dq_region" else ws_bytes
    assert (ws.numpy(np.uint8, (ws_bytes + 64,))[left:] == 0x5A).all(), "bytes of the workspace, or behind it, were written"
    return got[off:off + count]


@pytest.mark.gpu
@pytest.mark.parametrize("geo", [(128, 1, 28, 28, 10, 5, 5, 0, 0, 1, 1),    # 73728 positions: a thread has all channels
                                 (64, 1, 28, 28, 10, 5, 5, 0, 0, 1, 1),     # two groups of threads, five channels each
                                 (40, 4, 28, 28, 17, 3, 3, 1, 1, 1, 1),     # two groups of 9 and 8 channels, padded windows of 12 rows
                                 (3, 1, 9, 11, 16, 2, 3, 0, 0, 1, 1),       # 216 positions: four groups, the last wavefronts past the end
                                 (1, 3, 7, 9, 15, 4, 4, 3, 2, 1, 2),        # rows whose first taps are outside, all of them or some
                                 (2, 7, 6, 6, 20, 3, 3, 4, 4, 1, 1),        # 21 rows of 3, windows wholly outside
                                 (2, 1, 8, 8, 47, 8, 8, 4, 4, 1, 1),        # 8 rows of 8, the last group with 11 of 12 channels
                                 (1, 2, 5, 5, 3, 6, 5, 1, 0, 1, 1),         # 12 rows of 5, fewer than four channels
                                 (1, 1, 2, 4, 5, 2, 4, 0, 0, 1, 1),         # the input is one window
                                 (1, 1, 1, 5, 5, 1, 5, 0, 2, 1, 1),         # an input shorter than a load of 8 bytes
                                 (2, 1, 4, 12, 6, 3, 9, 0, 1, 1, 1),        # rows of more than 8 taps
                                 (3, 1, 9, 11, 16, 2, 2, 0, 0, 1, 1),       # rows of two taps
                                 (1, 2, 5, 5, 3, 4, 5, 0, 0, 1, 1)])        # 8 rows of 5, fewer than four channels
def test_conv2dq_direct_rows(gpu, ob, geo):
    """Windows of at most 64 taps, read row by row: loads that reach past the input's ends, the threads that share a position."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo))
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    Ho, Wo = ob.conv_out_hw(H, W, kh, kw, ph, pw, sh, sw)
    bias = rng.integers(-9999, 9999, Ho * Wo).astype(np.int32)
    want_y, want_acc = ob.conv2dq_forward(geo, x, w, [0.02, 0.013, 0.9], [17, 250, 100], bias=bias)
    y, acc = gpu.conv2dq_host(geo, x, w, [0.02, 0.013, 0.9], [17, 250, 100], bias=bias, want_acc=True)
    assert gpu.last_kernel() == "conv2dq_direct"
    assert np.array_equal(acc, want_acc) and np.array_equal(y, want_y)


PIXEL_GEOS = [(1, 16, 8, 8, 32, 3, 3, 1, 1, 1, 1),       # one tile, whole chunks
              (3, 17, 5, 7, 33, 3, 3, 1, 1, 1, 1),       # 35 positions an image, a channel past a chunk, one past a tile
              (5, 1, 1, 3, 2, 1, 3, 0, 1, 1, 1),         # images of three pixels
              (2, 20, 9, 11, 65, 5, 5, 2, 2, 2, 2),      # stride 2, 30 positions an image
              (1, 70, 13, 9, 100, 3, 5, 0, 2, 2, 1),     # two blocks of channels, the second nearly empty, oblong window
              (4, 64, 16, 16, 130, 3, 3, 1, 1, 1, 1),    # whole k-steps, stores of 16 positions
              (2, 250, 6, 6, 40, 1, 1, 0, 0, 1, 1),      # 1 x 1, no border
              (2, 130, 7, 7, 48, 5, 5, 2, 2, 1, 1),      # a long reduction
              (9, 6, 12, 10, 64, 4, 2, 3, 0, 3, 2)]      # borders above and below only, wider than the window reaches


@pytest.mark.parametrize("tile", [1, 2, 3, 4, 5, 6])
@pytest.mark.parametrize("geo", PIXEL_GEOS)
def test_conv2dq_pixels_tiles_vs_oracle(gpu, ob, geo, tile):
    """The two-launch route, every tile forced: remainders of positions, channels, chunks and k-steps, images that end inside a
    group of 16 positions, tensors on and off their alignment, all zero-point forms and both epilogues."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo) + tile)
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    Ho, Wo = ob.conv_out_hw(H, W, kh, kw, ph, pw, sh, sw)
    gpu.set_option("conv_variant", 10 + tile)
    try:
        for i, (sc, zp, with_bias) in enumerate((([1 / 255, 0.01, 0.05], [0, 128, 128], False), ([0.02, 0.013, 0.9], [17, 250, 100], True),
                                                 ([1.5, 1.0, 1.0], [200, 3, 9], True))):
            bias = rng.integers(-9999, 9999, Ho * Wo).astype(np.int32) if with_bias else None
            want, _ = ob.conv2dq_forward(geo, x, w, sc, zp, bias=bias)
            got = conv2dq_at(gpu, geo, x, w, sc, zp, bias, i)
            assert gpu.last_kernel() == "conv2dq_pixels", (geo, tile, zp, gpu.last_kernel())
            assert np.array_equal(got.reshape(want.shape), want), (geo, tile, zp)
    finally:
        gpu.set_option("conv_variant", 0)


REGION_GEOS = [(1, 16, 8, 16, 32, 3, 3, 1, 1, 1, 1),      # whole chunks, one block of channels
               (3, 17, 5, 7, 33, 3, 3, 1, 1, 1, 1),       # a channel past a chunk, one past a block; rows shorter than a load
               (2, 1, 9, 21, 10, 5, 5, 0, 0, 1, 1),       # one channel, an odd number of chunks
               (2, 20, 19, 11, 65, 5, 5, 2, 2, 2, 2),     # stride 2, a second group with one channel
               (1, 70, 13, 9, 100, 3, 5, 0, 2, 2, 1),     # five chunks, oblong window, columns the windows do not reach
               (3, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1),     # bands of one row, 56 of a block's 64 positions
               (2, 250, 6, 6, 40, 1, 1, 0, 0, 1, 1),      # 1 x 1, no border
               (1, 33, 40, 37, 64, 3, 3, 1, 1, 1, 1),     # odd rows, three chunks
               (5, 6, 12, 10, 64, 4, 2, 3, 0, 3, 2),      # rows above and below the image, wider than the window reaches
               (2, 12, 64, 100, 48, 5, 5, 2, 2, 1, 1)]    # more weights in a row than in a chunk, bands of few rows


@pytest.mark.parametrize("geo", REGION_GEOS)
def test_conv2dq_region_vs_oracle(gpu, ob, geo):
    """The band in LDS, forced: remainders of positions, channels, chunks and k-steps, bands that end early, tensors on and off their
    alignment, all zero-point forms and both epilogues; the workspace is not touched."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo) + 3)
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    Ho, Wo = ob.conv_out_hw(H, W, kh, kw, ph, pw, sh, sw)
    gpu.set_option("conv_variant", 20)
    try:
        for i, (sc, zp, with_bias) in enumerate((([1 / 255, 0.01, 0.05], [0, 128, 128], False), ([0.02, 0.013, 0.9], [17, 250, 100], True),
                                                 ([1.5, 1.0, 1.0], [200, 3, 9], True), ([1.5, 1.0, 1.0], [7, 128, 9], True))):
            bias = rng.integers(-9999, 9999, Ho * Wo).astype(np.int32) if with_bias else None
            want, _ = ob.conv2dq_forward(geo, x, w, sc, zp, bias=bias)
            got = conv2dq_at(gpu, geo, x, w, sc, zp, bias, i)
            assert gpu.last_kernel() == "conv2dq_region", (geo, zp, gpu.last_kernel())
            assert np.array_equal(got.reshape(want.shape), want), (geo, zp)
    finally:
        gpu.set_option("conv_variant", 0)


# Layers with enough images for bands of many rows: blocks of 64 channels a wavefront, several of them and several staging tiles one
# after another (the bands are asserted in test_launches.py); and 1 x 1 windows, whose weights are ordered four channels at a time.
REGION_TALL_GEOS = [(32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1),     # 7 rows: 7 blocks of 64 x 64
                    (64, 16, 112, 112, 60, 3, 3, 1, 1, 2, 2),   # 14 rows: 13 blocks, 26 staging tiles, four rows of weights empty
                    (64, 16, 56, 56, 32, 3, 3, 1, 1, 1, 1),     # 14 rows: 13 blocks of 64 x 32
                    (64, 15, 57, 55, 29, 3, 3, 1, 1, 1, 1),     # 15 rows and a last band of 12, weights byte by byte
                    (40, 14, 111, 109, 70, 3, 3, 1, 1, 2, 2),   # 13 staging tiles, a second group of six channels
                    (2, 64, 14, 14, 40, 1, 1, 0, 0, 1, 1),      # 1 x 1: whole chunks, 24 rows of weights empty
                    (2, 20, 13, 15, 33, 1, 1, 0, 0, 1, 1),      # a chunk of four channels, a last band of three rows
                    (3, 48, 28, 28, 100, 1, 1, 0, 0, 1, 1),     # three chunks: half of the last k-step is empty
                    (64, 48, 28, 28, 120, 1, 1, 0, 0, 1, 1)]    # the same in bands of 14 rows


@pytest.mark.parametrize("geo", REGION_TALL_GEOS)
def test_conv2dq_region_of_tall_bands_vs_oracle(gpu, ob, geo):
    """As above; the oracle computes the first, a middle and the last image, and a run with the images moved by one has to agree."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo) + 4)
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    Ho, Wo = ob.conv_out_hw(H, W, kh, kw, ph, pw, sh, sw)
    some = sorted({0, N // 2, N - 1})
    bias = rng.integers(-9999, 9999, Ho * Wo).astype(np.int32)
    gpu.set_option("conv_variant", 20)
    try:
        for i, (sc, zp, b) in enumerate((([0.02, 0.013, 0.9], [17, 128, 100], None), ([0.02, 0.013, 0.9], [17, 250, 100], bias))):
            want, _ = ob.conv2dq_forward((len(some),) + geo[1:], np.ascontiguousarray(x[some]), w, sc, zp, bias=b)
            got = conv2dq_at(gpu, geo, x, w, sc, zp, b, i).reshape(N, Cout, Ho, Wo)
            assert gpu.last_kernel() == "conv2dq_region", (geo, zp, gpu.last_kernel())
            assert np.array_equal(got[some], want.reshape(len(some), Cout, Ho, Wo)), (geo, zp)
            turned = conv2dq_at(gpu, geo, np.roll(x, 1, axis=0), w, sc, zp, b, 1 - i).reshape(N, Cout, Ho, Wo)
            assert np.array_equal(np.roll(got, 1, axis=0), turned), (geo, zp)
    finally:
        gpu.set_option("conv_variant", 0)


@pytest.mark.parametrize("geo", [(8, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1), (8, 116, 24, 24, 25, 3, 3, 1, 1, 1, 1), (3, 134, 30, 31, 70, 5, 5, 2, 2, 1, 1),
                                 (6, 100, 33, 35, 60, 3, 3, 1, 1, 2, 2), (24, 17, 64, 64, 96, 1, 1, 0, 0, 1, 1)])
def test_conv2dq_layers_the_library_sends_to_the_two_launches(gpu, ob, geo):
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo))
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    sc, zp = [0.02, 0.013, 0.02 * np.sqrt(Cin * kh * kw)], [17, 125, 100]
    want, _ = ob.conv2dq_forward(geo, x, w, sc, zp)
    got = conv2dq_at(gpu, geo, x, w, sc, zp, None, 0)
    assert gpu.last_kernel() == "conv2dq_pixels", gpu.last_kernel()
    assert np.array_equal(got.reshape(want.shape), want)


@pytest.mark.parametrize("geo,kern", [((8, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1), "conv2dq_pixels"),        # the band kernel could take it
                                      ((24, 17, 64, 64, 96, 1, 1, 0, 0, 1, 1), "conv2dq_pixels"),       # 17 taps, 96 channels
                                      ((16, 1024, 14, 14, 256, 1, 1, 0, 0, 1, 1), "conv2dq_pixels"),    # long windows on small maps
                                      ((32, 64, 56, 56, 64, 3, 3, 1, 1, 1, 1), "conv2dq_region"),
                                      ((11, 36, 14, 14, 32, 3, 3, 1, 1, 1, 1), "conv2dq_band"),
                                      ((64, 10, 12, 12, 20, 5, 5, 0, 0, 1, 1), "conv2dq_image"),
                                      ((40, 4, 28, 28, 17, 3, 3, 1, 1, 1, 1), "conv2dq_direct")])
def test_conv2dq_leaves_the_workspace_alone(gpu, ob, geo, kern):
    """Layers that have a kernel of one launch: the workspace keeps its bytes, and may be null, whatever the layer runs as."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo))
    x = rng.integers(0, 256, (N, Cin, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (Cout, Cin, kh, kw), dtype=np.uint8)
    qp = gpu.qparams3([0.02, 0.013, 0.02 * np.sqrt(Cin * kh * kw)], [17, 125, 100])
    want, want_acc = ob.conv2dq_forward(geo, x, w, [0.02, 0.013, 0.02 * np.sqrt(Cin * kh * kw)], [17, 125, 100])
    D, l = gpu.DeviceBuffer, gpu.lib()
    size = int(l.lten_hip_conv2dq_workspace_bytes(*geo))
    dx, dw, ws, dy, dacc = D.from_numpy(x), D.from_numpy(w), D(size), D(want.size), D(4 * want.size)
    gpu.check(l.lten_hip_fill_u8(ws.ptr, size, 0x5A))
    for memory in (ws.ptr, None):
        gpu.check(l.lten_hip_fill_u8(dy.ptr, want.size, 0xA5))
        gpu.check(l.lten_hip_conv2dq_forward(*geo, dx.ptr, dw.ptr, None, qp, dy.ptr, memory))
        assert gpu.last_kernel() == kern
        assert np.array_equal(dy.numpy(np.uint8, want.shape), want)
        gpu.check(l.lten_hip_conv2dq_forward_acc(*geo, dx.ptr, dw.ptr, None, qp, dacc.ptr, memory))
        assert np.array_equal(dacc.numpy(np.int32, want.shape), want_acc)
    assert (ws.numpy(np.uint8, (size,)) == 0x5A).all(), "the workspace was written"


def test_conv2dq_pixels_in_groups_of_images(gpu, ob):
    """605 MB of pixels: the library's 512 MB hold seven of the nine images."""
    geo = (9, 1, 2048, 2048, 2, 3, 3, 1, 1, 1, 1)
    rng = np.random.default_rng(9)
    x = rng.integers(0, 256, (9, 1, 2048, 2048), dtype=np.uint8)
    w = rng.integers(0, 256, (2, 1, 3, 3), dtype=np.uint8)
    want, _ = ob.conv2dq_forward(geo, x, w, [0.02, 0.013, 0.06], [17, 125, 100])
    D = gpu.DeviceBuffer
    dx, dw, dy = D.from_numpy(x), D.from_numpy(w), D(want.size)
    gpu.set_option("conv_variant", 12)
    try:
        gpu.check(gpu.lib().lten_hip_conv2dq_forward(*geo, dx.ptr, dw.ptr, None, gpu.qparams3([0.02, 0.013, 0.06], [17, 125, 100]), dy.ptr, None))
        assert gpu.last_kernel() == "conv2dq_pixels"
    finally:
        gpu.set_option("conv_variant", 0)
    assert np.array_equal(dy.numpy(np.uint8, want.shape), want)


def test_conv2dq_pixels_take_turns(gpu, ob):
    """4 to 24 MB of pixels have three places that calls take in turn: calls one behind the other on inputs of their own, and two
    recorded ones replayed between them."""
    geo = (34, 16, 90, 90, 48, 1, 1, 0, 0, 1, 1)
    rng = np.random.default_rng(34)
    sc, zp = [0.02, 0.013, 0.06], [17, 125, 100]
    w = rng.integers(0, 256, (48, 16, 1, 1), dtype=np.uint8)
    xs = [rng.integers(0, 256, geo[:4], dtype=np.uint8) for _ in range(4)]
    want = [ob.conv2dq_forward(geo, x, w, sc, zp)[0] for x in xs]
    D, l, qp = gpu.DeviceBuffer, gpu.lib(), gpu.qparams3(sc, zp)
    dw, dxs, dys = D.from_numpy(w), [D.from_numpy(x) for x in xs], [D(want[0].size) for _ in xs]
    call = lambda i: gpu.check(l.lten_hip_conv2dq_forward(*geo, dxs[i].ptr, dw.ptr, None, qp, dys[i].ptr, None))
    gpu.set_option("conv_variant", 12)
    try:
        call(0)
        with gpu.Graph() as g:
            call(0)
            call(1)
        assert gpu.last_kernel() == "conv2dq_pixels"
        for rep in range(4):
            for dy in dys:
                gpu.check(l.lten_hip_fill_u8(dy.ptr, want[0].size, rep))
            call(2)
            g.launch()
            call(3)
            for i in range(4):
                assert np.array_equal(dys[i].numpy(np.uint8, want[i].shape), want[i]), (rep, i)
    finally:
        gpu.set_option("conv_variant", 0)
