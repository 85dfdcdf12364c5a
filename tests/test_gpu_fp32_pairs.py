"""The fp32 GEMM tiles on fp16 pairs (csrc/sgemm_pairs.hip): tile and k-step edges in every layout, the folds of long sums, operands
that are left to the bf16 tiles, where the tiles are the default, and a recorded launch."""
import numpy as np
import pytest

from test_gpu_fp32_tiles import sgemm

pytestmark = pytest.mark.gpu

PAIRS = 41
NAME = "sgemm_fast_128x128_pairs"


@pytest.mark.parametrize("tA,tB", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("M,N,K", [(131, 133, 16 * 5 + 7), (64, 58, 48), (128, 256, 1), (257, 130, 16 * 33 + 5), (140, 129, 16 * 64), (1100, 1030, 40), (130, 133, 4100)])
def test_edges_in_all_layouts(gpu, M, N, K, tA, tB):
    """Partial tiles and k-steps, one k-step, a fold after 512 of K, rows too long to be held.  Integers: exact.  alpha, beta, padded odd rows."""
    rng = np.random.default_rng(M + K + 2 * tA + tB)
    A = rng.integers(-8, 9, (M, K)).astype(np.float32)
    B = rng.integers(-8, 9, (K, N)).astype(np.float32)
    want = A @ B
    assert np.array_equal(sgemm(gpu, tA, tB, A, B, PAIRS, pad=3), want)
    assert gpu.last_kernel() == NAME
    assert np.array_equal(sgemm(gpu, tA, tB, A, B, PAIRS, 2.0, -1.0, want, pad=1, shift=4), want)


def bound(A, B):
    """What sums of fp32 products may lose: (K + 8) roundings of 2^-23 of the sum of magnitudes (the pieces lose 2^-21 of a product at most)."""
    return (A.shape[1] + 8) * 2.0 ** -23 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64))


@pytest.mark.parametrize("tA,tB", [(0, 0), (1, 1)])
def test_operands_left_to_the_bf16_tiles(gpu, tA, tB):
    """Infinities and NaN; rows whose values span more than fp16 does, against columns without their large ones; beta: what a marked tile
    adds to is added to once."""
    rng = np.random.default_rng(5)
    M, N, K = 300, 290, 70
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = rng.standard_normal((K, N)).astype(np.float32)
    C0 = rng.standard_normal((M, N)).astype(np.float32)
    wide, cols = A.copy(), B.copy()
    wide[130, :] *= np.float32(2.0 ** -60)
    wide[130, 0] = 1e10
    cols[0, :200] = 0  # of row 130 only the small values count there
    got = sgemm(gpu, tA, tB, wide, cols, PAIRS, 1.0, 1.0, C0)
    want = wide.astype(np.float64) @ cols.astype(np.float64)
    # (adding C0 rounds once more, by 2^-24 of the result)
    assert (np.abs(got - (want + C0)) <= bound(wide, cols) + 2.0 ** -23 * np.abs(want + C0)).all()
    got = sgemm(gpu, tA, tB, wide, cols, PAIRS)
    assert (np.abs(got - want) <= bound(wide, cols)).all()
    A[3, 5], A[77, 1], B[9, 100] = np.inf, np.nan, -np.inf
    got = sgemm(gpu, tA, tB, A, B, PAIRS)
    with np.errstate(all="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    Af, Bf = np.where(np.isfinite(A), A, 0), np.where(np.isfinite(B), B, 0)
    assert (np.abs(got[fine] - want[fine]) <= bound(Af, Bf)[fine]).all()


@pytest.mark.parametrize("ea,eb", [(-130, 40), (90, 5), (-60, -60), (0, 0)])
def test_rows_of_any_magnitude(gpu, ea, eb):
    """Rows and columns 2^20 apart from each other, denormal and near the largest ones among them, zero rows and columns between."""
    rng = np.random.default_rng(ea + 200)
    M, N, K = 200, 150, 90
    A = (rng.standard_normal((M, K)) * 2.0 ** (ea + rng.integers(-10, 11, (M, 1)))).astype(np.float32)
    B = (rng.standard_normal((K, N)) * 2.0 ** (eb + rng.integers(-10, 11, (1, N)))).astype(np.float32)
    A[7], B[:, 9] = 0, 0
    want = A.astype(np.float64) @ B.astype(np.float64)
    for tA, tB in ((0, 1), (1, 0)):
        got = sgemm(gpu, tA, tB, A, B, PAIRS)
        # (results below the normal range are rounded at 2^-149)
        assert (np.abs(got - want) <= bound(A, B) + 2.0 ** -149).all()


def test_denormal_results_round_once_each(gpu):
    rng = np.random.default_rng(1)
    A = rng.integers(1, 9, (130, 1)).astype(np.float32)
    B = (rng.integers(1, 9, (1, 131)) * 2.0 ** -149).astype(np.float32)
    assert np.array_equal(sgemm(gpu, 0, 0, A, B, PAIRS), A @ B)


@pytest.mark.parametrize("K", [1025, 2048, 4096])
def test_no_more_error_than_the_bf16_tiles(gpu, K):
    """2-norm error against float64 on N(0, 1): below that of the 128 x 128 bf16 tiles, whose sums round K / 8 times."""
    rng = np.random.default_rng(K)
    A, B = rng.standard_normal((600, K)).astype(np.float32), rng.standard_normal((K, 600)).astype(np.float32)
    want = A.astype(np.float64) @ B.astype(np.float64)
    err = [np.linalg.norm(sgemm(gpu, 0, 1, A, B, t) - want) for t in (PAIRS, 21)]
    assert err[0] <= err[1], err


def test_default_for_large_products(gpu):
    """A fully connected layer's forward with bias and relu, a stack, and a launch graph that replays the route."""
    rng = np.random.default_rng(2)
    D, l = gpu.DeviceBuffer, gpu.lib()
    M, fin, fout = 3001, 2060, 3075
    x = rng.integers(-4, 5, (M, fin)).astype(np.float32)
    w = rng.integers(-4, 5, (fout, fin)).astype(np.float32)
    b = rng.integers(-9, 10, fout).astype(np.float32)
    dX, dW, dB, dY, dR = D.from_numpy(x), D.from_numpy(w), D.from_numpy(b), D(4 * M * fout), D(4 * M * fout)
    gpu.check(l.lten_hip_fc_forward_relu_f32(M, fin, fout, dX.ptr, dW.ptr, dB.ptr, dY.ptr, dR.ptr))
    assert gpu.last_kernel() == NAME
    want = x @ w.T + b
    assert np.array_equal(dY.numpy(np.float32, want.shape), want) and np.array_equal(dR.numpy(np.float32, want.shape), np.maximum(want, 0))
    with gpu.Graph() as g:
        gpu.check(l.lten_hip_fc_forward_f32(M, fin, fout, dX.ptr, dW.ptr, dB.ptr, dY.ptr))
    for step in range(3):
        x = np.roll(x, 1, axis=0)
        dX.upload(x)
        dR.upload(np.zeros((M, fout), np.float32))
        gpu.check(l.lten_hip_fc_forward_f32(M, fin, fout, dX.ptr, dW.ptr, dB.ptr, dR.ptr))
        g.launch()
        assert np.array_equal(dY.numpy(np.float32, want.shape), x @ w.T + b)
        assert np.array_equal(dR.numpy(np.float32, want.shape), x @ w.T + b)
    # a stack, the right operand shared or not
    S, M, N, K = 3, 1100, 1300, 1200
    A = rng.integers(-4, 5, (S, M, K)).astype(np.float32)
    B = rng.integers(-4, 5, (S, N, K)).astype(np.float32)
    dA, dB, dC = D.from_numpy(A), D.from_numpy(B), D(4 * S * M * N)
    gpu.set_option("sgemm_tile", PAIRS)
    try:
        for stride_b, right in ((N * K, B), (0, B[[0, 0, 0]])):
            gpu.check(l.lten_hip_sgemm_strided_batched(0, 1, M, N, K, 1.0, dA.ptr, K, M * K, dB.ptr, K, stride_b, 0.0, dC.ptr, N, M * N, S))
            assert np.array_equal(dC.numpy(np.float32, (S, M, N)), A @ right.transpose(0, 2, 1))
    finally:
        gpu.set_option("sgemm_tile", 0)
