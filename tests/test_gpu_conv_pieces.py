"""Conv2d on the bf16 matrix cores (csrc/conv_split.hip, csrc/conv_split_wgrad.hip) at the sizes where it can go wrong: every tile on maps whose tiles
cross rows, images and column strips, ragged channels, strides with their classes of pixels; values without three bf16
pieces; a recorded launch graph."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES = 7


def out_hw(geo):
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    return (H + 2 * ph - kh) // sh + 1, (W + 2 * pw - kw) // sw + 1


def forward64(geo, x, w, bias):
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    Ho, Wo = out_hw(geo)
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    y = np.zeros((N, Cout, Ho, Wo)) + bias[None, :, None, None]
    with np.errstate(all="ignore"):
        for i in range(kh):
            for j in range(kw):
                xs = xp[:, :, i:i + (Ho - 1) * sh + 1:sh, j:j + (Wo - 1) * sw + 1:sw]
                for c in range(Cin):
                    y += w[None, :, c, i, j, None, None].astype(np.float64) * xs[:, None, c]
    return y


def dgrad64(geo, w, dy):
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    Ho, Wo = out_hw(geo)
    dx = np.zeros((N, Cin, max(H + 2 * ph, (Ho - 1) * sh + kh), max(W + 2 * pw, (Wo - 1) * sw + kw)))
    for i in range(kh):
        for j in range(kw):
            dx[:, :, i:i + (Ho - 1) * sh + 1:sh, j:j + (Wo - 1) * sw + 1:sw] += np.einsum("oc,nohw->nchw", w[:, :, i, j].astype(np.float64), dy.astype(np.float64))
    return dx[:, :, ph:ph + H, pw:pw + W]


def run(gpu, geo, x, w, bias, dy, variant):
    """y and dx (None where the tile does not take the shape)."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    D, l = gpu.DeviceBuffer, gpu.lib()
    dX, dW, dB, dDY = (D.from_numpy(t) for t in (x, w, bias, dy))
    Y, DX = D.from_numpy(np.full(dy.shape, 7, np.float32)), D.from_numpy(np.full(x.shape, 7, np.float32))
    ws = D(max(int(l.lten_hip_conv2d_dgrad_workspace_bytes(*geo)), 16))
    gpu.set_option("conv_variant", variant)
    try:
        gpu.check(l.lten_hip_conv2d_forward_f32(*geo, dX.ptr, dW.ptr, dB.ptr, Y.ptr))
        fk = gpu.last_kernel()
        gpu.check(l.lten_hip_conv2d_dgrad_f32(*geo, dW.ptr, dDY.ptr, DX.ptr, ws.ptr))
        dk = gpu.last_kernel()
    finally:
        gpu.set_option("conv_variant", 0)
    y = Y.numpy(np.float32, dy.shape) if fk == "conv2d_pieces_forward" else None
    return y, (DX.numpy(np.float32, x.shape) if dk == "conv2d_pieces_dgrad" else None)


@pytest.mark.parametrize("geo", [
    (3, 20, 14, 14, 70, 3, 3, 1, 1, 1, 1),     # tiles across rows and images, ragged channels both ways
    (2, 33, 28, 28, 64, 5, 5, 2, 2, 1, 1),     # 25 taps, a chunk of one channel
    (1, 48, 17, 130, 96, 3, 3, 1, 1, 1, 1),    # two column strips of 65
    (1, 8, 9, 300, 33, 3, 2, 1, 1, 1, 1),      # three strips or more, the last one narrower; an oblong window
    (4, 32, 13, 29, 40, 3, 3, 1, 1, 2, 2),     # stride 2: four classes of pixels, odd map
    (3, 40, 12, 10, 65, 4, 3, 2, 0, 2, 2),     # stride 2, oblong window, a class with other paddings
    (9, 16, 8, 8, 33, 3, 3, 3, 3, 1, 1),       # more padding than the window is wide
    (1, 16, 1, 1, 32, 3, 3, 1, 1, 1, 1),       # a single pixel
    (70, 17, 5, 5, 31, 2, 2, 0, 0, 1, 1),      # many images to a tile
])
def test_every_tile_on_integers(gpu, geo):
    """Exact in any order; each tile by itself where it takes the shape, and the one the library picks."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo))
    mk = lambda *s: rng.integers(-8, 9, s).astype(np.float32)
    x, w, bias, dy = mk(N, Cin, H, W), mk(Cout, Cin, kh, kw), mk(Cout), mk(N, Cout, *out_hw(geo))
    want_y, want_dx = forward64(geo, x, w, bias), dgrad64(geo, w, dy)
    taken = 0
    for variant in [10] + [11 + k for k in range(TILES)]:
        y, dx = run(gpu, geo, x, w, bias, dy, variant)
        taken += (y is not None) + (dx is not None)
        assert y is None or np.array_equal(y, want_y), (geo, variant)
        assert dx is None or np.array_equal(dx, want_dx), (geo, variant)
    assert taken >= 4


def wgrad64(geo, x, dy):
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    Ho, Wo = out_hw(geo)
    xp = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (ph, ph), (pw, pw)))
    dw = np.empty((Cout, Cin, kh, kw))
    with np.errstate(all="ignore"):
        for i in range(kh):
            for j in range(kw):
                xs = xp[:, :, i:i + (Ho - 1) * sh + 1:sh, j:j + (Wo - 1) * sw + 1:sw]
                for c in range(Cin):
                    dw[:, c, i, j] = (dy.astype(np.float64) * xs[:, None, c]).sum(axis=(0, 2, 3))
    return dw


def run_wgrad(gpu, geo, x, dy, pieces=True):
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    D, l = gpu.DeviceBuffer, gpu.lib()
    dX, dDY, DW = D.from_numpy(x), D.from_numpy(dy), D.from_numpy(np.full((Cout, Cin, kh, kw), 7, np.float32))
    ws = D(max(int(l.lten_hip_conv2d_wgrad_workspace_bytes(*geo)), 16))
    gpu.set_option("conv_variant", 10)
    try:
        gpu.check(l.lten_hip_conv2d_wgrad_f32(*geo, dX.ptr, dDY.ptr, DW.ptr, ws.ptr))
        assert (gpu.last_kernel() == "conv2d_pieces_wgrad") == pieces, gpu.last_kernel()
    finally:
        gpu.set_option("conv_variant", 0)
    return DW.numpy(np.float32, (Cout, Cin, kh, kw))


@pytest.mark.parametrize("geo", [
    (16, 33, 7, 7, 65, 3, 3, 1, 1, 1, 1),      # chunks of eight rows across images, ragged channels in clamped loads
    (2, 8, 3, 4, 9, 3, 3, 1, 1, 1, 1),         # fewer pixels than a chunk
    (3, 70, 30, 32, 130, 3, 3, 2, 1, 1, 1),    # row padding 2, three blocks of output channels
    (2, 40, 9, 96, 33, 3, 3, 0, 1, 1, 1),      # two strips
    (1, 31, 5, 66, 63, 3, 3, 1, 1, 1, 1),      # 66 columns: an octet of two
    (2, 34, 6, 9, 20, 3, 3, 1, 0, 1, 1),       # no column padding; the last values of both tensors in partial loads
    (3, 64, 57, 57, 64, 3, 3, 1, 1, 2, 2),     # stride 2 on an odd map
    (2, 34, 20, 19, 66, 3, 3, 0, 0, 2, 2),     # stride 2 without padding
    (40, 7, 6, 5, 3, 3, 3, 1, 1, 2, 2),        # stride 2, many small images
    # what a thread stages, slot by slot: 15 and 18 and 20 slots to a chunk at stride two, the last a slot at the end of x; rows
    # of one and of nine columns
    (2, 33, 29, 57, 65, 3, 3, 1, 1, 2, 2), (3, 17, 21, 21, 40, 3, 3, 1, 1, 2, 2), (2, 31, 14, 15, 33, 3, 3, 1, 1, 2, 2),
    (5, 32, 7, 1, 33, 3, 3, 1, 1, 2, 2), (4, 33, 9, 9, 20, 3, 3, 1, 1, 1, 1), (3, 40, 6, 1, 40, 3, 3, 1, 1, 1, 1),
])
def test_weight_gradient_on_integers(gpu, geo):
    """Exact in any order."""
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    rng = np.random.default_rng(sum(geo))
    x = rng.integers(-8, 9, (N, Cin, H, W)).astype(np.float32)
    dy = rng.integers(-8, 9, (N, Cout, *out_hw(geo))).astype(np.float32)
    assert np.array_equal(run_wgrad(gpu, geo, x, dy), wgrad64(geo, x, dy))


@pytest.mark.parametrize("geo", [(2, 1, 2, 1, 3, 3, 3, 1, 1, 1, 1), (3, 1, 2, 1, 3, 3, 3, 1, 1, 1, 1), (4, 1, 2, 1, 3, 3, 3, 1, 1, 1, 1),
                                 (2, 1, 2, 2, 3, 3, 3, 1, 1, 2, 2)])
def test_weight_gradient_of_tensors_that_end_in_two_slots_of_a_thread(gpu, geo):
    """Two rows within the last three values of x, both staged by one thread: left to the other routes."""
    rng = np.random.default_rng(3)
    x, dy = rng.integers(-8, 9, geo[:4]).astype(np.float32), rng.integers(-8, 9, (geo[0], geo[4], *out_hw(geo))).astype(np.float32)
    assert np.array_equal(run_wgrad(gpu, geo, x, dy, pieces=False), wgrad64(geo, x, dy))


@pytest.mark.parametrize("stride", [1, 2])
def test_weight_gradient_rounding_and_values_without_three_pieces(gpu, stride):
    geo = (2, 20, 13, 14, 40, 3, 3, 1, 1, stride, stride)
    Ho, Wo = out_hw(geo)
    rng = np.random.default_rng(6)
    x, dy = rng.standard_normal((2, 20, 13, 14)).astype(np.float32), rng.standard_normal((2, 40, Ho, Wo)).astype(np.float32)
    terms = 2 * Ho * Wo + 8

    def close(got, want, bound):
        fine = np.isfinite(want)
        return (np.abs(got[fine] - want[fine]) <= bound[fine]).all()

    assert close(run_wgrad(gpu, geo, x, dy), wgrad64(geo, x, dy), terms * 2.0 ** -23 * wgrad64(geo, np.abs(x), np.abs(dy)))
    tiny, big = (x * 2.0 ** -130).astype(np.float32), dy * np.float32(2.0 ** 40)
    assert close(run_wgrad(gpu, geo, tiny, big), wgrad64(geo, tiny, big), terms * 2.0 ** -23 * wgrad64(geo, np.abs(tiny), np.abs(big)))
    x[0, 3, 0, 5], dy[1, 39, Ho - 1, Wo - 1] = np.inf, np.nan
    x[1, 0, 6, 6] = 3.4e38
    dy[1] *= 0.05
    got, want = run_wgrad(gpu, geo, x, dy), wgrad64(geo, x, dy)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    mag = wgrad64(geo, np.where(np.isfinite(x), np.abs(x), 0), np.where(np.isfinite(dy), np.abs(dy), 0))
    assert close(got, want, terms * 2.0 ** -23 * mag)


def test_rounding(gpu):
    """Random values: at most (terms + 8) roundings of 2^-23 of the sum of magnitudes."""
    geo = (2, 24, 19, 19, 40, 3, 3, 1, 1, 1, 1)
    rng = np.random.default_rng(1)
    x, w = rng.standard_normal((2, 24, 19, 19)).astype(np.float32), rng.standard_normal((40, 24, 3, 3)).astype(np.float32)
    bias, dy = rng.standard_normal(40).astype(np.float32), rng.standard_normal((2, 40, 19, 19)).astype(np.float32)
    y, dx = run(gpu, geo, x, w, bias, dy, 10)
    assert (np.abs(y - forward64(geo, x, w, bias)) <= (24 * 9 + 9) * 2.0 ** -23 * forward64(geo, np.abs(x), np.abs(w), np.abs(bias))).all()
    assert (np.abs(dx - dgrad64(geo, w, dy)) <= (40 * 9 + 8) * 2.0 ** -23 * dgrad64(geo, np.abs(w), np.abs(dy))).all()


@pytest.mark.parametrize("tile", [2, 4, 5, 6, 7])
def test_sums_of_the_small_tiles_round_once_a_k_step(gpu, tile):
    """As in the GEMM tiles: 0.41 sqrt(n) 2^-24 in the 2-norm for n k-steps of 16 channels."""
    geo = (1, 256, 16, 16, 40, 3, 3, 1, 1, 1, 1)
    rng = np.random.default_rng(tile)
    x, w = rng.standard_normal(geo[:4]).astype(np.float32), rng.standard_normal((40, 256, 3, 3)).astype(np.float32)
    bias, dy = np.zeros(40, np.float32), np.zeros((1, 40, 16, 16), np.float32)
    y, _ = run(gpu, geo, x, w, bias, dy, 10 + tile)
    want = forward64(geo, x, w, bias)
    err = np.linalg.norm(y - want) / np.linalg.norm(want)
    assert err <= 0.5 * np.sqrt(256 * 9 / 16) * 2.0 ** -24, err


@pytest.mark.parametrize("where", ["x", "w"])
def test_values_without_three_pieces(gpu, where):
    """Infinities, NaN and values that round to an infinite bf16 reach the outputs they reach in a sum of fp32 products;
    denormals against large values keep their precision."""
    geo = (2, 20, 11, 12, 40, 3, 3, 1, 1, 1, 1)
    rng = np.random.default_rng(5)
    x, w = rng.standard_normal((2, 20, 11, 12)).astype(np.float32), rng.standard_normal((40, 20, 3, 3)).astype(np.float32)
    bias, dy = np.zeros(40, np.float32), rng.standard_normal((2, 40, 11, 12)).astype(np.float32)
    if where == "x":
        x[0, 3, 0, 5], x[1, 19, 10, 11], x[1, 0, 5, 5] = np.inf, np.nan, 3.4e38
        w[:, 0] *= 0.05
    else:
        w[3, 4, 1, 1], w[39, 19, 2, 0] = -np.inf, 3.4e38
        x[:, 19] *= 0.05
    want = forward64(geo, x, w, bias)
    y, _ = run(gpu, geo, x, w, bias, dy, 16)
    assert np.array_equal(np.isnan(y), np.isnan(want)) and np.array_equal(np.isposinf(y), np.isposinf(want)) and np.array_equal(np.isneginf(y), np.isneginf(want))
    fine = np.isfinite(want)
    mag = forward64(geo, np.where(np.isfinite(x), np.abs(x), 0), np.where(np.isfinite(w), np.abs(w), 0), bias)
    assert (np.abs(y[fine] - want[fine]) <= ((20 * 9 + 8) * 2.0 ** -23 * mag)[fine]).all()
    x, w = rng.standard_normal(x.shape).astype(np.float32), rng.standard_normal(w.shape).astype(np.float32)
    if where == "x":
        x, w = (x * 2.0 ** -130).astype(np.float32), w * np.float32(2.0 ** 40)
    else:
        x, w = x * np.float32(2.0 ** 40), (w * 2.0 ** -130).astype(np.float32)
    y, _ = run(gpu, geo, x, w, bias, dy, 16)
    assert (np.abs(y - forward64(geo, x, w, bias)) <= (20 * 9 + 8) * 2.0 ** -23 * forward64(geo, np.abs(x), np.abs(w), bias)).all()


@pytest.mark.parametrize("tile", range(1, TILES + 1))
def test_a_large_bias_is_rounded_in_once(gpu, tile):
    """A bias 2^20 times the products: the sum's own roundings and one more of the result."""
    geo = (2, 24, 19, 19, 40, 3, 3, 1, 1, 1, 1)
    rng = np.random.default_rng(tile)
    x, w = rng.standard_normal((2, 24, 19, 19)).astype(np.float32), rng.standard_normal((40, 24, 3, 3)).astype(np.float32)
    bias, dy = (rng.standard_normal(40) * 2.0 ** 20).astype(np.float32), np.zeros((2, 40, 19, 19), np.float32)
    y, _ = run(gpu, geo, x, w, bias, dy, 10 + tile)
    want, zero = forward64(geo, x, w, bias), np.zeros_like(bias)
    assert (np.abs(y - want) <= (24 * 9 + 8) * 2.0 ** -23 * forward64(geo, np.abs(x), np.abs(w), zero) + 2.0 ** -24 * np.abs(want)).all()


@pytest.mark.parametrize("q", range(70, 76))
def test_weight_gradient_whose_halves_add_up_past_the_scaled_range(gpu, q):
    """Each half of a chunk's k-steps sums to just below 2^80, which the pieces' factors take to just below infinity; exact."""
    geo = (1, 40, 16, 16, 33, 3, 3, 1, 1, 1, 1)
    x, dy = np.full(geo[:4], 1.5 * 2.0 ** 40, np.float32), np.full((1, 33, 16, 16), 2.0 ** (q - 40), np.float32)
    assert np.array_equal(run_wgrad(gpu, geo, x, dy), wgrad64(geo, x, dy))


@pytest.mark.parametrize("tile", [1, 3, 6])
@pytest.mark.parametrize("geo", [(2, 20, 11, 13, 40, 3, 3, 1, 1, 2, 2),     # a stride on an odd map: four classes of pixels
                                 (1, 18, 5, 150, 34, 3, 3, 1, 1, 1, 1),     # two strips of columns
                                 (2, 20, 12, 11, 70, 3, 5, 1, 0, 1, 1)])    # an oblong window, padding past it in the data gradient
def test_infinities_in_strides_strips_and_the_data_gradient(gpu, geo, tile):
    """Infinities, NaN and values from 2^103 on in x and dy touch the outputs they touch in a sum of fp32 products, no others."""
    rng = np.random.default_rng(tile)
    x, w = rng.standard_normal(geo[:4]).astype(np.float32), rng.standard_normal((geo[4], geo[1], *geo[5:7])).astype(np.float32)
    bias, dy = rng.standard_normal(geo[4]).astype(np.float32), rng.standard_normal((geo[0], geo[4], *out_hw(geo))).astype(np.float32)
    w *= 0.02
    for t in (x, dy):
        t[0, 3, 0, 5], t[-1, -1, -1, -1], t[-1, 0, 2, 2] = -np.inf, np.nan, 3.4e38
    y, dx = run(gpu, geo, x, w, bias, dy, 10 + tile)
    taps = geo[5] * geo[6]
    for got, of, terms in ((y, lambda a, b, c: forward64(geo, a, b, c), geo[1] * taps), (dx, lambda a, b, c: dgrad64(geo, b, a), geo[4] * taps)):
        if got is None:
            continue
        t = x if got is y else dy
        with np.errstate(all="ignore"):
            want = of(t, w, bias)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
        fine = np.isfinite(want)
        mag = of(np.where(np.isfinite(t), np.abs(t), 0), np.abs(w), np.abs(bias))
        assert (np.abs(got[fine] - want[fine]) <= ((terms + 8) * 2.0 ** -23 * mag)[fine]).all()
    assert y is not None or dx is not None


@pytest.mark.parametrize("low", [-110, -130, -140])
@pytest.mark.parametrize("stride", [1, 2])
def test_values_of_wide_range_side_by_side(gpu, stride, low):
    """Every other channel (forward, data gradient) or column (weight gradient) is near or below the smallest normal and meets
    large values of the other operand: each term counts to its own last bits."""
    geo = (2, 20, 11, 12, 40, 3, 3, 1, 1, stride, stride)
    rng = np.random.default_rng(low + 300 + stride)
    normal = lambda *s: rng.standard_normal(s)

    def pair(a, b, at_a, at_b):   # odd indexes of a small, those of b large
        ia, ib = [slice(None)] * a.ndim, [slice(None)] * b.ndim
        for t, i, at, odd, even in ((a, ia, at_a, low, 0), (b, ib, at_b, 100, -40)):
            i[at] = slice(1, None, 2)
            t[tuple(i)] *= 2.0 ** odd
            i[at] = slice(0, None, 2)
            t[tuple(i)] *= 2.0 ** even
        return a.astype(np.float32), b.astype(np.float32)

    Ho, Wo = out_hw(geo)
    zero, x, dy = np.zeros(40, np.float32), normal(2, 20, 11, 12), normal(2, 40, Ho, Wo)
    x32, w32 = pair(x.copy(), normal(40, 20, 3, 3), 1, 1)
    y, _ = run(gpu, geo, x32, w32, zero, dy.astype(np.float32), 10)
    assert (np.abs(y - forward64(geo, x32, w32, zero)) <= (20 * 9 + 8) * 2.0 ** -23 * forward64(geo, np.abs(x32), np.abs(w32), zero)).all()
    dy32, w32 = pair(dy.copy(), normal(40, 20, 3, 3), 1, 0)
    _, dx = run(gpu, geo, x.astype(np.float32), w32, zero, dy32, 10)
    assert (np.abs(dx - dgrad64(geo, w32, dy32)) <= (40 * 9 + 8) * 2.0 ** -23 * dgrad64(geo, np.abs(w32), np.abs(dy32))).all()
    dy32, x32 = pair(dy.copy(), x.copy(), 3, 3)
    if stride == 2:   # (x columns 2 wo - 1 .. 2 wo + 1: large ones under every other output column's centre tap)
        x32 = x.copy()
        x32[..., 0::4] *= 2.0 ** -40
        x32[..., 2::4] *= 2.0 ** 100
        x32 = x32.astype(np.float32)
    dw = run_wgrad(gpu, geo, x32, dy32)
    assert (np.abs(dw - wgrad64(geo, x32, dy32)) <= (2 * Ho * Wo + 8) * 2.0 ** -23 * wgrad64(geo, np.abs(x32), np.abs(dy32))).all()


def test_inside_a_recorded_launch_graph(gpu):
    """The packed weights and the slices' sums live in memory of the library: a layer that ran before is recorded with these tiles and replays to
    the eager values with new inputs."""
    geo = (8, 64, 24, 24, 64, 3, 3, 1, 1, 1, 1)
    D, l = gpu.DeviceBuffer, gpu.lib()
    rng = np.random.default_rng(2)
    x, w, dy = D(4 * 8 * 64 * 576), D(4 * 64 * 64 * 9), D(4 * 8 * 64 * 576)
    y, dx, dw = D(4 * 8 * 64 * 576), D(4 * 8 * 64 * 576), D(4 * 64 * 64 * 9)
    ws = D(max(int(l.lten_hip_conv2d_dgrad_workspace_bytes(*geo)), int(l.lten_hip_conv2d_wgrad_workspace_bytes(*geo))))
    names = []

    def fill():
        for buf in (x, w, dy):
            buf.upload(rng.standard_normal(buf.nbytes // 4).astype(np.float32))

    def step():
        gpu.check(l.lten_hip_conv2d_forward_f32(*geo, x.ptr, w.ptr, None, y.ptr)); names.append(gpu.last_kernel())
        gpu.check(l.lten_hip_conv2d_dgrad_f32(*geo, w.ptr, dy.ptr, dx.ptr, ws.ptr)); names.append(gpu.last_kernel())
        gpu.check(l.lten_hip_conv2d_wgrad_f32(*geo, x.ptr, dy.ptr, dw.ptr, ws.ptr)); names.append(gpu.last_kernel())

    gpu.set_option("conv_variant", 10)
    try:
        fill()
        step()
        with gpu.Graph() as graph:
            step()
        assert names == ["conv2d_pieces_forward", "conv2d_pieces_dgrad", "conv2d_pieces_wgrad"] * 2, names
        for _ in range(3):
            fill()
            step()
            want = [b.numpy(np.float32, (b.nbytes // 4,)).copy() for b in (y, dx, dw)]
            for b in (y, dx, dw):
                gpu.check(l.lten_hip_zero(b.ptr, b.nbytes))
            graph.launch()
            for b, v in zip((y, dx, dw), want):
                assert np.array_equal(b.numpy(np.float32, v.shape), v)
    finally:
        gpu.set_option("conv_variant", 0)


@pytest.mark.parametrize("geo,entry,kernel", [
    ((32, 128, 28, 28, 256, 3, 3, 1, 1, 2, 2), "dgrad", "conv2d_pieces_dgrad"),              # columns 71 to 80 us, this 56
    ((20, 144, 56, 56, 416, 3, 3, 1, 1, 2, 2), "dgrad", "conv2d_dgrad_batched_gemm_col2im"),  # 194, on pieces 236
    ((30, 176, 14, 14, 320, 5, 5, 2, 2, 1, 1), "wgrad", "conv2d_wgrad_columns_gemm"),        # implicit GEMM 325 us, this 172
    ((44, 144, 21, 21, 375, 5, 5, 2, 2, 2, 2), "wgrad", "conv2d_wgrad_columns_gemm"),        # 303, 137
    ((32, 256, 14, 14, 512, 3, 3, 1, 1, 2, 2), "wgrad", "conv2d_wgrad_columns_gemm"),        # on pieces 70, 53
])
def test_routes_by_the_gemms_own_estimate(gpu, geo, entry, kernel):
    """Layers that estimates of slower GEMM tiles sent to a kernel of up to twice the time; the result on integers, exact."""
    rng = np.random.default_rng(sum(geo))
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    Ho, Wo = out_hw(geo)
    D, l = gpu.DeviceBuffer, gpu.lib()
    dy = rng.integers(-2, 3, (N, Cout, Ho, Wo)).astype(np.float32)
    if entry == "dgrad":
        t, shape, ws = rng.integers(-2, 3, (Cout, Cin, kh, kw)).astype(np.float32), geo[:4], l.lten_hip_conv2d_dgrad_workspace_bytes(*geo)
    else:
        t, shape, ws = rng.integers(-2, 3, geo[:4]).astype(np.float32), (Cout, Cin, kh, kw), l.lten_hip_conv2d_wgrad_workspace_bytes(*geo)
    dT, dDY, out, work = D.from_numpy(t), D.from_numpy(dy), D(4 * int(np.prod(shape))), D(max(int(ws), 16))
    gpu.check(getattr(l, f"lten_hip_conv2d_{entry}_f32")(*geo, dT.ptr, dDY.ptr, out.ptr, work.ptr))
    assert gpu.last_kernel() == kernel, gpu.last_kernel()
    got = out.numpy(np.float32, shape)
    # a part of the outputs, enough to see a wrong operand: two images, or two input channels
    want = dgrad64((2, *geo[1:]), t, dy[:2]) if entry == "dgrad" else wgrad64((N, 2, *geo[2:]), t[:, :2], dy)
    assert np.array_equal(got[:2] if entry == "dgrad" else got[:, :2], want)


@pytest.mark.parametrize("N,Cin,Cout", [(4, 130, 250), (8, 97, 257), (6, 512, 64), (2, 256, 256)])
def test_weight_gradient_of_wide_layers_on_integers(gpu, N, Cin, Cout):
    """16 tiles and more, so 16 slices or fewer: channels that are no multiple of 3, 4, 32 or 64; one to 16 slices.  Exact."""
    geo = (N, Cin, 10, 12, Cout, 3, 3, 1, 1, 1, 1)
    rng = np.random.default_rng(Cin + Cout)
    x, dy = rng.integers(-8, 9, (N, Cin, 10, 12)).astype(np.float32), rng.integers(-8, 9, (N, Cout, 10, 12)).astype(np.float32)
    xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1)))
    want = np.stack([dy.transpose(1, 0, 2, 3).reshape(Cout, -1) @ xp[:, :, i:i + 10, j:j + 12].transpose(0, 2, 3, 1).reshape(-1, Cin)
                     for i in range(3) for j in range(3)], axis=-1)
    assert np.array_equal(run_wgrad(gpu, geo, x, dy).reshape(Cout, Cin, 9), want)


@pytest.mark.parametrize("geo", [
    (5, 16, 1, 3, 32, 3, 3, 1, 1, 1, 1),       # planes of fewer values than a quad: staged from a copy
    (2, 48, 2, 2, 40, 3, 3, 1, 1, 1, 1),       # every quad of a plane reaches past one of its ends; an odd number of chunks
    (2, 64, 5, 6, 33, 3, 3, 2, 2, 1, 1),       # quads turned by two and more; rows and their padding no multiple of 4
    (12, 90, 7, 7, 70, 3, 3, 1, 1, 1, 1),      # narrow maps: more positions to a tile than pixels, tiles of fewer than 256 pixels
    (20, 20, 33, 33, 40, 5, 5, 2, 2, 2, 2),    # a window and stride that fit with narrow strips or small tiles only
    (3, 16, 31, 43, 64, 3, 3, 0, 0, 2, 2),     # 3 x 3 at stride 2, one chunk, no padding
    (9, 20, 22, 22, 13, 5, 5, 4, 2, 2, 2),     # tiles of 122 pixels
    (5, 33, 40, 41, 35, 3, 3, 1, 1, 2, 2),     # tiles of 75 and 133 pixels, strips of columns
    (30, 18, 5, 9, 33, 7, 7, 3, 3, 1, 1),      # whole images to a tile
])
def test_patches_of_quads_on_integers(gpu, geo):
    """The quads at the ends of a plane, patches that do not fit at a full tile, one chunk to six.  Exact in any order."""
    rng = np.random.default_rng(sum(geo))
    N, Cin, H, W, Cout, kh, kw, ph, pw, sh, sw = geo
    mk = lambda *s: rng.integers(-8, 9, s).astype(np.float32)
    x, w, bias, dy = mk(N, Cin, H, W), mk(Cout, Cin, kh, kw), mk(Cout), mk(N, Cout, *out_hw(geo))
    want_y, want_dx = forward64(geo, x, w, bias), dgrad64(geo, w, dy)
    taken = 0
    for variant in [10] + [11 + k for k in range(TILES)]:
        y, dx = run(gpu, geo, x, w, bias, dy, variant)
        taken += (y is not None) + (dx is not None)
        assert y is None or np.array_equal(y, want_y), (geo, variant)
        assert dx is None or np.array_equal(dx, want_dx), (geo, variant)
    assert taken >= 8


@pytest.mark.parametrize("geo", [
    (3, 6, 1, 1, 4, 3, 3, 1, 1, 1, 1), (2, 11, 1, 2, 70, 3, 3, 1, 1, 1, 1),  # quads that reach over the planes behind, at the end of either tensor
    (5, 2, 3, 1, 3, 3, 3, 1, 1, 2, 2), (2, 9, 2, 5, 5, 3, 3, 1, 1, 2, 2),
    (6, 4, 17, 17, 33, 3, 3, 1, 1, 1, 1), (6, 1, 17, 18, 33, 3, 3, 1, 1, 2, 2),  # few channels: the others repeat the last
    (7, 37, 4, 40, 66, 3, 3, 1, 1, 2, 2), (9, 40, 5, 13, 20, 3, 3, 1, 0, 2, 2),  # up to 20 slots: the second kind of a lane
])
def test_weight_gradient_staging_on_integers(gpu, geo):
    """Loads that leave a plane, a row or the tensor, both strides.  Exact in any order."""
    rng = np.random.default_rng(sum(geo))
    x = rng.integers(-8, 9, geo[:4]).astype(np.float32)
    dy = rng.integers(-8, 9, (geo[0], geo[4], *out_hw(geo))).astype(np.float32)
    assert np.array_equal(run_wgrad(gpu, geo, x, dy), wgrad64(geo, x, dy))


@pytest.mark.parametrize("entry", ["forward", "dgrad"])
def test_planes_of_less_than_a_quad_in_groups_of_images(gpu, entry):
    """2100 images of 16384 planes of one value: the copy that they are staged from holds 2048 images at a time.  Exact in any order
    (a window meets a plane with its centre tap only)."""
    N, C, M = 2100, 16384, 40
    rng = np.random.default_rng(N)
    t = rng.integers(-8, 9, (N, C), dtype=np.int8).astype(np.float32)
    w = rng.integers(-8, 9, (M, C, 3, 3) if entry == "forward" else (C, M, 3, 3), dtype=np.int8).astype(np.float32)
    bias = rng.integers(-8, 9, M).astype(np.float32)
    D, l = gpu.DeviceBuffer, gpu.lib()
    dT, dW, dB, out = D.from_numpy(t), D.from_numpy(w), D.from_numpy(bias), D.from_numpy(np.full((N, M), 7, np.float32))
    gpu.set_option("conv_variant", 10)
    try:
        if entry == "forward":
            gpu.check(l.lten_hip_conv2d_forward_f32(N, C, 1, 1, M, 3, 3, 1, 1, 1, 1, dT.ptr, dW.ptr, dB.ptr, out.ptr))
        else:
            geo = (N, M, 1, 1, C, 3, 3, 1, 1, 1, 1)
            ws = D(max(int(l.lten_hip_conv2d_dgrad_workspace_bytes(*geo)), 16))
            gpu.check(l.lten_hip_conv2d_dgrad_f32(*geo, dW.ptr, dT.ptr, out.ptr, ws.ptr))
        assert gpu.last_kernel() == f"conv2d_pieces_{entry}"
    finally:
        gpu.set_option("conv_variant", 0)
    want = t @ w[:, :, 1, 1].T + bias if entry == "forward" else t @ w[:, :, 1, 1]
    assert np.array_equal(out.numpy(np.float32, (N, M)), want)
