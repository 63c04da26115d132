"""fp32 results on the bf16 matrix cores (mtc_gemm_f32, k_gemm_f32; run on an MI355X): X and the
weights cut into bf16 planes, at every tile height's edges, and values that have no such planes."""

import numpy as np
import pytest

from oracle import mtc_oracle as O
from tensorpack_amd.core.quadtree import QTAllocation
from tensorpack_amd.kernels.gemm import MTCMatrix

from conftest import cell_format_matrices, leaf_matrix, tile_rows

pytestmark = pytest.mark.gpu

# (K, N): a partial last K-step and column tile; many K-steps (split K, several per block)
SHAPES = {"ragged": (992, 288), "deep": (4096, 544)}


@pytest.fixture(scope="module")
def mats():
    return cell_format_matrices(SHAPES)


def _tol(K):
    # each output: sums of 16 rows of K, rounded once to fp32 (a random walk of half-ulp steps on the running sum);
    # held to six of them, as if every plane pair went to the one accumulator
    return (np.sqrt(6 * K / 16) + 2) * 2.0 ** -25


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("form", ["qt", "qtp", "p16", "uniform"])
def test_f32_tiles_at_every_height(gpu, mats, shape, form):
    import torch
    m, W_hat = mats[shape, form]
    K = W_hat.shape[0]
    t = m.device_tiles(gpu)
    heights = set()
    for M in (1, 17, 31, 32, 33, 64, 65, 100, 128, 129, 250) + ((700, 703, 2999, 3000, 3009) if shape == "ragged" else ()):
        print("f32 split", shape, form, M, flush=True)
        heights.add(tile_rows(t, M, True))
        X = (np.random.RandomState(M).randn(M, K) * np.exp(3 * np.random.RandomState(K).randn(K))).astype(np.float32)
        Y = t.gemm_f32(torch.from_numpy(X).to(gpu)).cpu().numpy()
        err = O.relative_frobenius_error(O.qt_gemm_f64(X, W_hat), Y)
        assert err <= _tol(K), (M, err)
    assert heights == ({32, 64, 128} if shape == "ragged" else {32, 64})


@pytest.mark.parametrize("form", ["qt", "qtp", "uniform"])
@pytest.mark.parametrize("M,rows", [(20, 32), (64, 32), (100, 32), (700, 64), (3000, 128)])
def test_f32_tiles_infinities_nan_and_range(gpu, mats, form, M, rows):
    """Infinities and NaN go where the fp64 product has them, the other rows keep their values; finite
    values near the end of fp32's range (the scaled planes would be infinite) give finite results, and
    subnormal ones lose nothing but the rounding of subnormal sums. Blocks of every height, whose plain
    fp32 pass takes 1 to 8 turns."""
    import torch
    m, W_hat = mats["ragged", form]
    K = W_hat.shape[0]
    t = m.device_tiles(gpu)
    assert tile_rows(t, M, True) == rows
    X = np.random.RandomState(M).randn(M, K).astype(np.float32)
    Z = X.copy()
    Z[3, 5], Z[7, 100], Z[M - 1, K - 1] = np.inf, np.nan, -np.inf
    print("f32 split non-finite", form, M, flush=True)
    Y = t.gemm_f32(torch.from_numpy(Z).to(gpu)).cpu().numpy()
    with np.errstate(invalid="ignore"):
        ref = Z.astype(np.float64) @ W_hat.astype(np.float64)
    assert np.array_equal(np.isnan(Y), np.isnan(ref)) and np.array_equal(np.isinf(Y), np.isinf(ref))
    assert np.array_equal(np.sign(Y[np.isinf(Y)]), np.sign(ref[np.isinf(ref)]))
    rest = np.setdiff1d(np.arange(M), [3, 7, M - 1])
    assert O.relative_frobenius_error(ref[rest], Y[rest]) <= np.sqrt(K) * 2.0 ** -25    # an fma chain of K steps
    big = np.zeros((M, K), np.float32)
    big[np.arange(M), np.arange(M) % K] = np.float32(3.4e38)
    small = np.abs(W_hat[np.arange(M) % K]).max(axis=1, keepdims=True) < 0.99
    Yb = t.gemm_f32(torch.from_numpy(big).to(gpu)).cpu().numpy()
    with np.errstate(over="ignore"):
        want = (big.astype(np.float64) @ W_hat.astype(np.float64)).astype(np.float32)
    sel = small & np.isfinite(want)
    assert sel.any() and np.allclose(Yb[sel], want[sel], rtol=2.0 ** -22, atol=0)
    tiny = (X * 1e-38).astype(np.float32)
    Yt = t.gemm_f32(torch.from_numpy(tiny).to(gpu)).cpu().numpy().astype(np.float64)
    ref = tiny.astype(np.float64) @ W_hat.astype(np.float64)
    # the bar of the others on the largest output, and half a subnormal step for each of at most 32 partials and sums
    assert np.abs(Yt - ref).max() <= np.sqrt(K) * 2.0 ** -25 * np.abs(ref).max() + 32 * 2.0 ** -149


def _flat(W, P, scales, S=32):
    """A matrix of S x S leaves of one code width, with the given bf16 scales, and its W_hat."""
    K, N = W.shape
    leaf, modes = {S: np.ones((K // S, N // S), bool)}, {S: np.full((K // S, N // S), P)}
    a = QTAllocation((S,), leaf, modes, {S: scales}, None, K * N * P, weights=W)
    return MTCMatrix.from_quadtree(a), O.qt_dequant(W, (S,), leaf, modes, {S: scales})


@pytest.mark.parametrize("form", ["qt", "p16", "uniform"])
def test_f32_same_signed_sums(gpu, form):
    """Sums of one sign over 8192 rows that are not split: two, two or three and three weight planes. The
    small plane products must not fall below half an ulp of the running sum, which loses them all to one side."""
    import torch
    K, N, M = 8192, 2048, 4096
    rng = np.random.RandomState(5)
    W = (0.5 + rng.rand(K, N)).astype(np.float32)
    if form == "uniform":
        s = np.exp(-4.4 + 0.1 * rng.rand(K // 32, N // 32)).astype(np.float32)
        m = MTCMatrix.from_allocation(W, np.full((K // 32, N // 32), 8, np.uint8), s, 32)
        W_hat = O.uniform_to_array(W, np.full((K // 32, N // 32), 8, np.uint8), s, 32)
    else:
        m, W_hat = _flat(W, 16 if form == "p16" else 8, np.full((K // 32, N // 32), 2.0 ** (-14 if form == "p16" else -6), np.float32))
    t = m.device_tiles(gpu)
    X = torch.from_numpy((0.5 + rng.rand(M, K)).astype(np.float32)).to(gpu)
    print("f32 same-signed", form, flush=True)
    Y = t.gemm_f32(X).double()
    ref = X.double() @ torch.from_numpy(W_hat).to(gpu).double()
    # rounded once per 16 rows of K (one MFMA), each time by up to half an ulp of the running sum: a random walk
    assert ((Y - ref).norm() / ref.norm()).item() <= (np.sqrt(K / 16) + 2) * 2.0 ** -24
    assert abs(((Y - ref).mean() / ref.mean()).item()) <= 2.0 ** -24       # to neither side


@pytest.mark.parametrize("form", ["qt", "p16", "uniform"])
def test_f32_single_products(gpu, form):
    """One non-zero X a row: every output is one product, right to its own rounding and the sum of the small
    plane products' (some are left out below 2^-30). Mantissas whose middle and low planes are as large as
    they get."""
    import torch
    K = N = 256
    if form == "qt":                       # 79 * 209 = 0x407F: two planes, the second 0xFE
        W = np.full((K, N), 79 * 209 * 2.0 ** -14, np.float32)
        m, W_hat = _flat(W, 8, np.full((8, 8), 209 * 2.0 ** -14, np.float32))
    elif form == "p16":                    # 20382 * 209 = 0x40FFFE: three planes
        W = np.full((K, N), 20382 * 209 * 2.0 ** -22, np.float32)
        m, W_hat = _flat(W, 16, np.full((8, 8), 209 * 2.0 ** -22, np.float32))
    else:
        s = np.full((8, 8), np.float32(0x80FFFF * 2.0 ** -23) / np.float32(127), np.float32)
        W = np.full((K, N), np.float32(127) * s[0, 0], np.float32)
        m = MTCMatrix.from_allocation(W, np.full((8, 8), 8, np.uint8), s, 32)
        W_hat = O.uniform_to_array(W, np.full((8, 8), 8, np.uint8), s, 32)
    low = W_hat.view(np.uint32) & 0xFFFF
    assert (low >= 0xFE00).all()                                           # the planes the test is about
    t = m.device_tiles(gpu)
    for M in (20, 64, 200):
        X = np.zeros((M, K), np.float32)
        X[np.arange(M), np.arange(M) % K] = np.array([0x3F80FFFF, 0xBFFFFFFF], np.uint32).view(np.float32)[np.arange(M) % 2]
        print("f32 single products", form, M, flush=True)
        Y = t.gemm_f32(torch.from_numpy(X).to(gpu)).cpu().numpy()
        ref = X.astype(np.float64) @ W_hat.astype(np.float64)
        # half an ulp of the result, and half an ulp of each of the sums of the small pairs: they are below 2^-6 of it
        assert (np.abs(Y - ref) <= np.abs(ref) * (2.0 ** -24 + 8 * 2.0 ** -30)).all(), np.abs(Y / ref - 1).max()


@pytest.mark.parametrize("form", ["qt", "qtp", "p16", "uniform"])
def test_f32_small_magnitudes(gpu, mats, form):
    """Normal fp32 inputs whose low bf16 planes would be below bf16's range, and such weights, cost no bits."""
    import torch
    m, W_hat = mats["ragged", form]
    K = W_hat.shape[0]
    t = m.device_tiles(gpu)
    for M in (17, 64, 100):
        X = np.random.RandomState(M).randn(M, K).astype(np.float32)
        for e in (-100, -112, -116, -120):
            Xe = (X * 2.0 ** e).astype(np.float32)
            print("f32 small magnitudes", form, M, e, flush=True)
            Y = t.gemm_f32(torch.from_numpy(Xe).to(gpu)).cpu().numpy()
            up = 2.0 ** -e                     # exact in 64 bits: the error function's floor is far above these values
            assert O.relative_frobenius_error(O.qt_gemm_f64(Xe, W_hat) * up, Y.astype(np.float64) * up) <= _tol(K), (M, e)
    if form == "uniform":
        rng = np.random.RandomState(9)
        W = (rng.randn(K, 288) * 2.0 ** -112).astype(np.float32)
        modes = np.full((K // 32, 9), 8, np.uint8)
        s = (np.exp(0.1 * rng.rand(K // 32, 9)) * 2.0 ** -117).astype(np.float32)
        w, W_hat = MTCMatrix.from_allocation(W, modes, s, 32).device_tiles(gpu), O.uniform_to_array(W, modes, s, 32)
        Y = w.gemm_f32(torch.from_numpy(X).to(gpu)).cpu().numpy()
        up = 2.0 ** 112
        assert O.relative_frobenius_error(O.qt_gemm_f64(X, W_hat) * up, Y.astype(np.float64) * up) <= _tol(K)


def test_f32_x_rows_far_apart(gpu):
    """X rows so far apart that 128 or 64 of them span 4 GiB: the call takes a lower tile, in the workspace of its
    usual plan."""
    import torch
    K = N = 4096
    M = 250
    t = leaf_matrix("qt", K, N, 3)[0].device_tiles(gpu)
    assert tile_rows(t, M, True) == 128
    X = torch.randn(M, K, device=gpu)
    want = X.double() @ t.dequant().double()
    for ldx in ((1 << 23) + 4, (1 << 24) + 4):
        print("f32 far rows", ldx, flush=True)
        Z = torch.empty(M * ldx, device=gpu).as_strided((M, K), (ldx, 1))
        Z.copy_(X)
        Y = t.gemm_f32(Z).double()
        assert ((Y - want).norm() / want.norm()).item() <= _tol(K), ldx
        del Z


@pytest.mark.parametrize("form", ["qt", "qtp", "p16", "uniform"])
def test_f32_large_sums(gpu, mats, form):
    """Finite sums past 2^80, which overflow the scaled accumulators: those tiles come from the plain pass."""
    import torch
    m, W_hat = mats["ragged", form]
    K = W_hat.shape[0]
    t = m.device_tiles(gpu)
    for M in (20, 700, 3000):
        X = np.random.RandomState(M).randn(M, K).astype(np.float32)
        X[: M // 2] *= np.float32(2.0 ** 90)
        print("f32 large sums", form, M, flush=True)
        Y = t.gemm_f32(torch.from_numpy(X).to(gpu)).cpu().numpy()
        ref = X.astype(np.float64) @ W_hat.astype(np.float64)
        assert np.isfinite(Y).all()
        for rows in (slice(0, M // 2), slice(M // 2, M)):
            assert O.relative_frobenius_error(ref[rows], Y[rows]) <= np.sqrt(K) * 2.0 ** -25    # an fma chain of K steps
