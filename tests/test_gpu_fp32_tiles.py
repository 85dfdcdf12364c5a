"""The fp32 GEMM tiles on the bf16 matrix cores (csrc/sgemm_fast.hip) at the sizes where they can go wrong: every tile in
every layout around its edges and its k-step, reductions shorter than a k-step and cut into uneven slices, operands off
16-byte boundaries, the fused relu, and operands whose values have no three bf16 pieces."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TILES = {12: (256, 256), 13: (256, 128), 14: (128, 256), 21: (128, 128), 24: (128, 128), 31: (64, 64), 32: (64, 64), 33: (64, 64),
         34: (128, 64), 35: (64, 128)}


def sgemm(gpu, tA, tB, A, B, tile=0, alpha=1.0, beta=0.0, C0=None, pad=0, shift=0):
    """C = alpha op(A) op(B) + beta C0 for the plain matrices A [M][K], B [K][N]; rows `pad` floats longer, bases `shift` bytes in."""
    M, K = A.shape
    N = B.shape[1]
    As, Bs = (A.T if tA else A), (B.T if tB else B)
    hold = []
    for X in (As, Bs):
        Xp = np.full((X.shape[0], X.shape[1] + pad), 1e30, np.float32)
        Xp[:, :X.shape[1]] = X
        buf = gpu.DeviceBuffer(Xp.nbytes + shift)
        buf.upload(Xp, offset=shift)
        hold.append((buf, Xp.shape[1]))
    C = np.full((M, N + pad), 7.0, np.float32)
    if C0 is not None:
        C[:, :N] = C0
    dC = gpu.DeviceBuffer.from_numpy(C)
    gpu.set_option("sgemm_tile", tile)
    try:
        gpu.sgemm(tA, tB, M, N, K, alpha, hold[0][0].ptr + shift, hold[0][1], hold[1][0].ptr + shift, hold[1][1], beta, dC, N + pad)
    finally:
        gpu.set_option("sgemm_tile", 0)
    out = dC.numpy(np.float32, C.shape)
    assert (out[:, N:] == 7.0).all()
    return out[:, :N]


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("tile", sorted(TILES))
def test_tile_edges_in_all_layouts(gpu, tile, tA, tB):
    """One tile and a last one that is moved back inside the matrix (odd sizes), a reduction with a partial k-step; then fewer
    rows than the tile.  Integers: exact in any order.  alpha, beta, padded odd leading dimensions."""
    bm, bn = TILES[tile]
    rng = np.random.default_rng(tile * 4 + 2 * tA + tB)
    for M, N, K in ((bm + 3, bn + 5, 16 * 5 + 7), (bm // 2 - 2, bn // 2 - 6, 48), (bm, 2 * bn, 1)):
        A = rng.integers(-8, 9, (M, K)).astype(np.float32)
        B = rng.integers(-8, 9, (K, N)).astype(np.float32)
        want = A @ B
        got = sgemm(gpu, tA, tB, A, B, tile, pad=3)
        assert gpu.last_kernel().startswith("sgemm_fast"), gpu.last_kernel()
        assert np.array_equal(got, want), (M, N, K)
        assert np.array_equal(sgemm(gpu, tA, tB, A, B, tile, 2.0, -1.0, want, pad=1, shift=4), want), (M, N, K)


@pytest.mark.parametrize("tile", [12, 21, 33])
def test_all_significand_bits_count(gpu, tile):
    """Every piece of a value takes part: 24-bit integers times a permutation with signs come back bit for bit; and over a
    reduction of one k-step the error stays below what fp32 sums allow, (K + 8) roundings of 2^-23 (a piece product left away
    by mistake is 2^-17 or more of |a| |b|)."""
    rng = np.random.default_rng(tile)
    n = 160
    A = (rng.integers(1 << 23, 1 << 24, (n, n)) * rng.choice([-1, 1], (n, n))).astype(np.float32)
    P = np.zeros((n, n), np.float32)
    P[rng.permutation(n), np.arange(n)] = rng.choice([-1, 1], n)
    assert np.array_equal(sgemm(gpu, 0, 0, A, P, tile), A @ P)
    assert np.array_equal(sgemm(gpu, 1, 1, P, A, tile), P @ A)
    A, B = rng.standard_normal((n, 16)).astype(np.float32), rng.standard_normal((16, n)).astype(np.float32)
    err = np.abs(sgemm(gpu, 0, 0, A, B, tile) - A.astype(np.float64) @ B.astype(np.float64))
    assert (err <= 24 * 2.0 ** -23 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))).all()


@pytest.mark.parametrize("tile", [t for t in sorted(TILES) if t != 12])
def test_sums_round_once_a_k_step(gpu, tile):
    """n k-steps that each round the sum at that time by up to 2^-24 of it (a standard deviation of 2^-24 / sqrt 3), the sum
    growing with their square root: 0.41 sqrt(n) 2^-24 in the 2-norm.  Rounded by every piece product it would be 1.0."""
    rng = np.random.default_rng(tile)
    A, B = rng.standard_normal((150, 4096)).astype(np.float32), rng.standard_normal((4096, 140)).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    err = np.linalg.norm(sgemm(gpu, 0, 1, A, B, tile) - want) / np.linalg.norm(want)
    assert err <= 0.5 * np.sqrt(4096 / 16) * 2.0 ** -24, err


@pytest.mark.parametrize("tile", [12, 24, 33])
def test_operands_without_three_pieces(gpu, tile):
    """Infinities, NaN and values that round to an infinite bf16 give what a sum of fp32 products gives, and touch nothing but
    their rows and columns; rows of denormals against large columns keep their precision."""
    rng = np.random.default_rng(3)
    M, N, K = 300, 290, 70
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    clean = sgemm(gpu, 0, 0, A, B, tile)
    A[3, 5], A[77, 1], B[9, 100], A[299, 69] = np.inf, np.nan, -np.inf, 3.4e38
    B[69] *= 0.25
    clean[299] = 0
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    for tA, tB in ((0, 0), (1, 1)):
        got = sgemm(gpu, tA, tB, A, B, tile)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
        fine = np.isfinite(want)
        scale = np.abs(A[:, :]).astype(np.float64)
        scale[~np.isfinite(scale)] = 0
        bound = (K + 8) * 2.0 ** -23 * (scale @ np.where(np.isfinite(B), np.abs(B), 0).astype(np.float64))
        assert (np.abs(got[fine] - want[fine]) <= bound[fine]).all()
    tiny = (rng.standard_normal((M, K)) * 2.0 ** -130).astype(np.float32)
    tiny[::2] = rng.standard_normal((M // 2, K))
    big = (rng.standard_normal((K, N)) * 2.0 ** 40).astype(np.float32)
    want = tiny.astype(np.float64) @ big.astype(np.float64)
    bound = (K + 8) * 2.0 ** -23 * (np.abs(tiny).astype(np.float64) @ np.abs(big).astype(np.float64))
    for tA, tB in ((0, 0), (1, 1)):
        assert (np.abs(sgemm(gpu, tA, tB, tiny, big, tile) - want) <= bound).all()


@pytest.mark.parametrize("tile", sorted(TILES))
def test_rows_of_wide_range(gpu, tile):
    """Values near and below the smallest normal beside normal ones in the same rows, where the other operand is large: every
    term counts to its own last bits, (K + 8) roundings of 2^-23 of the sum of magnitudes."""
    rng = np.random.default_rng(tile)
    M, N, K = 150, 140, 50
    for low in (-110, -125, -130, -140):
        A, B = rng.standard_normal((M, K)), rng.standard_normal((K, N))
        A[:, 1::2] *= 2.0 ** low
        B[0::2] *= 2.0 ** -40
        B[1::2] *= 2.0 ** 100
        B[0] *= rng.random(N) < 0.5
        A, B = A.astype(np.float32), B.astype(np.float32)
        want = A.astype(np.float64) @ B.astype(np.float64)
        bound = (K + 8) * 2.0 ** -23 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))
        assert (np.abs(sgemm(gpu, 0, 0, A, B, tile) - want) <= bound).all(), low
        assert (np.abs(sgemm(gpu, 1, 1, B.T, A.T, tile) - want.T) <= bound.T).all(), low
    two = sgemm(gpu, 0, 0, np.float32([[1, 1.23 * 2.0 ** -125]]), np.float32([[2.0 ** -40], [1.35 * 2.0 ** 120]]), tile)
    assert abs(two[0, 0] / (2.0 ** -40 + 1.23 * 1.35 * 2.0 ** -5) - 1) < 2.0 ** -21


@pytest.mark.parametrize("tile", [12, 21, 33])
def test_sums_that_leave_the_scaled_range(gpu, tile):
    """Values from 2^103 and sums from 2^80 on (which the pieces' factors would take to infinity) come out as fp32 sums do."""
    rng = np.random.default_rng(tile)
    A, B = rng.standard_normal((70, 40)), rng.standard_normal((40, 66))
    for a, b in ((2.0 ** 110, 2.0 ** -60), (2.0 ** 45, 2.0 ** 45), (2.0 ** 60, 2.0 ** 60)):
        x, y = (A * a).astype(np.float32), (B * b).astype(np.float32)
        want = x.astype(np.float64) @ y.astype(np.float64)
        bound = (40 + 8) * 2.0 ** -23 * (np.abs(x).astype(np.float64) @ np.abs(y).astype(np.float64))
        assert (np.abs(sgemm(gpu, 0, 1, x, y, tile) - want) <= bound).all(), (a, b)


@pytest.mark.parametrize("tA,tB", [(0, 1), (1, 0)])
@pytest.mark.parametrize("M,N,K", [(130, 1030, 4100), (300, 520, 2311)])
def test_uneven_slices_of_a_long_reduction(gpu, M, N, K, tA, tB):
    """Few tiles under a long reduction: slices of whole k-steps, the last one shorter, added with alpha and beta in order."""
    rng = np.random.default_rng(K)
    A = rng.integers(-4, 5, (M, K)).astype(np.float32)
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    want = A @ B
    got = sgemm(gpu, tA, tB, A, B, pad=1)
    assert gpu.last_kernel() == "sgemm_split_k", gpu.last_kernel()
    assert np.array_equal(got, want)
    assert np.array_equal(sgemm(gpu, tA, tB, A, B, 0, 2.0, -1.0, want), want)


def test_relu_in_the_tiles_store(gpu):
    """relu and relu_backward ride on the tiles' store with the values of the separate calls, bit for bit."""
    rng = np.random.default_rng(8)
    D, l = gpu.DeviceBuffer, gpu.lib()
    M, n_in, n_out = 601, 520, 2060
    X, W = rng.standard_normal((M, n_in)).astype(np.float32), rng.standard_normal((n_out, n_in)).astype(np.float32)
    b, dY = rng.standard_normal(n_out).astype(np.float32), rng.standard_normal((M, n_out)).astype(np.float32)
    dX, dW, dB, dDY = (D.from_numpy(t) for t in (X, W, b, dY))
    y, r, y2, g, g2 = D(4 * M * n_out), D(4 * M * n_out), D(4 * M * n_out), D(4 * M * n_in), D(4 * M * n_in)
    gpu.check(l.lten_hip_fc_forward_relu_f32(M, n_in, n_out, dX.ptr, dW.ptr, dB.ptr, y.ptr, r.ptr))
    assert gpu.last_kernel().startswith("sgemm_fast"), gpu.last_kernel()
    gpu.check(l.lten_hip_fc_forward_f32(M, n_in, n_out, dX.ptr, dW.ptr, dB.ptr, y2.ptr))
    Y = y2.numpy(np.float32, (M, n_out))
    assert np.array_equal(y.numpy(np.float32, Y.shape), Y)
    assert np.array_equal(r.numpy(np.float32, Y.shape), np.maximum(Y, 0))
    gpu.check(l.lten_hip_fc_backward_relu_f32(M, n_in, n_out, dX.ptr, dW.ptr, dDY.ptr, dX.ptr, g.ptr, None, None))
    gpu.check(l.lten_hip_fc_backward_f32(M, n_in, n_out, dX.ptr, dW.ptr, dDY.ptr, g2.ptr, None, None))
    assert np.array_equal(g.numpy(np.float32, X.shape), np.where(X > 0, g2.numpy(np.float32, X.shape), 0))


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_leading_dimensions_of_millions(gpu, tA, tB):
    """Rows 2 M values apart in both operands (a slice of a wide matrix), 256 of them under one tile: still the tiles."""
    M, N, K, ld = 260, 70, 40, (1 << 21) + 1
    rng = np.random.default_rng(2 * tA + tB)
    A, B = rng.integers(-8, 9, (M, K)).astype(np.float32), rng.integers(-8, 9, (K, N)).astype(np.float32)
    bufs = []
    for X in (A.T if tA else A, B.T if tB else B):
        X = np.ascontiguousarray(X)
        buf = gpu.DeviceBuffer(4 * ((X.shape[0] - 1) * ld + X.shape[1]))
        for r in range(X.shape[0]):
            buf.upload(X[r], offset=4 * r * ld)
        bufs.append(buf)
    C = gpu.DeviceBuffer(4 * M * N)
    for tile in (12, 31):
        gpu.set_option("sgemm_tile", tile)
        try:
            gpu.sgemm(tA, tB, M, N, K, 1.0, bufs[0].ptr, ld, bufs[1].ptr, ld, 0.0, C, N)
        finally:
            gpu.set_option("sgemm_tile", 0)
        assert gpu.last_kernel().startswith("sgemm_fast"), gpu.last_kernel()
        assert np.array_equal(C.numpy(np.float32, (M, N)), A @ B)


@pytest.mark.parametrize("M,N,K,tA,tB", [(2048, 2048, 2048, 0, 1), (1500, 1700, 2060, 1, 0), (1100, 3001, 1301, 0, 0)])
def test_values_keep_all_their_bits_in_long_sums(gpu, M, N, K, tA, tB):
    """What the library itself picks for a product with a long reduction: values of 24 significand bits against a selection with
    signs come back bit for bit."""
    rng = np.random.default_rng(M + N + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    first, sign = rng.integers(0, K, N), rng.choice(np.float32([-1, 1]), N)
    B = np.zeros((K, N), np.float32)
    B[first, np.arange(N)] = sign
    assert np.array_equal(sgemm(gpu, tA, tB, A, B), A[:, first] * sign)
