"""GEMMs of 128-wide tiles, whose products are six bf16 partial products of the
operands' three-way split, at their edges: every operand order, ragged rows and
columns, padded rows, few and many K stages, values that the split cannot hold.
Bounds against float64: per element, the first-order bound of 6 K rounded
additions, 6 K 2^-24 sum |a||b|; over the matrix sqrt(K) 2^-24, which a chain of
K fp32 additions of random signs stays below; integers whose sums stay below
2^24 are exact whatever the order, and only if no partial product is left out."""
import numpy as np
import pytest

from gpuutil import DBuf, log

pytestmark = pytest.mark.gpu


def _gemm(dev, ta, tb, A, B, M, N, K, pad=0, alpha=1.0):
    """C = alpha op(A) op(B) with `pad` extra floats per operand row."""
    from goneuron_amd._lib import check, lib
    Ap, Bp = (np.pad(x, ((0, 0), (0, pad)), constant_values=np.nan) for x in (A, B))
    dA, dB, dC = DBuf(dev, Ap), DBuf(dev, Bp), DBuf(dev, np.zeros((M, N), np.float32))
    check(dev.h, lib().gn_gemm(dev.h, ta, tb, M, N, K, alpha, dA.p, Ap.shape[1], dB.p, Bp.shape[1], dC.p, N))
    return dC.get()


def _op(x, t):
    return x.T if t else x


# the contiguous extent of each operand is a multiple of 4, as that path needs
@pytest.mark.parametrize("ta,tb,M,N,K,pad", [
    (0, 1, 1601, 1543, 64, 0), (0, 1, 1665, 1537, 320, 4), (0, 0, 1537, 1668, 128, 0), (0, 0, 1601, 1540, 64, 8),
    (1, 0, 1604, 1540, 64, 0), (1, 0, 1540, 1668, 192, 4), (1, 1, 1604, 1537, 128, 4), (0, 1, 1536, 1792, 256, 0)])
def test_gemm_split(dev, ta, tb, M, N, K, pad):
    log(f"gemm ta={ta} tb={tb} {M}x{N}x{K} pad={pad}")
    rng = np.random.default_rng(M + N + K)
    A = (rng.normal(size=(K, M) if ta else (M, K)) * np.exp(rng.normal(size=(1, 1)))).astype(np.float32)
    B = rng.normal(size=(N, K) if tb else (K, N)).astype(np.float32)
    a, b = _op(A, ta).astype(np.float64), _op(B, tb).astype(np.float64)
    err = _gemm(dev, ta, tb, A, B, M, N, K, pad) - a @ b
    assert np.all(np.abs(err) <= 6 * K * 2.0 ** -24 * (np.abs(a) @ np.abs(b)))
    assert np.linalg.norm(err) <= np.sqrt(K) * 2.0 ** -24 * np.linalg.norm(a @ b)
    lim = (1 << 23) // K  # of a product: both wide, then 15 to 17 bits from either side
    for ma, mb in ((int(lim ** 0.5), int(lim ** 0.5)), (lim, 1), (1, lim)):
        A, B = rng.integers(-ma, ma + 1, A.shape), rng.integers(-mb, mb + 1, B.shape)
        got = _gemm(dev, ta, tb, A.astype(np.float32), B.astype(np.float32), M, N, K, pad)
        assert np.array_equal(got, (_op(A, ta).astype(np.float64) @ _op(B, tb)).astype(np.float32))


@pytest.mark.parametrize("ta,tb,M,N,K,pad", [
    (0, 1, 1601, 1543, 320, 0), (0, 1, 1536, 1792, 256, 0), (0, 0, 1601, 1540, 320, 8), (0, 0, 1537, 1668, 256, 0),
    (1, 0, 1604, 1540, 320, 0), (1, 0, 1540, 1668, 256, 4), (1, 1, 1604, 1537, 320, 4), (1, 1, 1604, 1540, 256, 0),
    (1, 0, 1604, 1540, 1088, 0)])
def test_gemm_split_from_five_stages(dev, ta, tb, M, N, K, pad):
    """The last K of the fp32 kernel and the first of the split, each order."""
    test_gemm_split(dev, ta, tb, M, N, K, pad)


def test_short_products_stay_on_fp32(dev):
    """Up to K = 256 a plain product has the bits of a linear Dense forward."""
    from goneuron_amd._lib import check, lib
    B, I, O = 1604, 256, 1600
    log("plain product of four K stages")
    rng = np.random.default_rng(9)
    x, W = rng.normal(size=(B, I)).astype(np.float32), rng.normal(size=(O, I)).astype(np.float32)
    dx, dw, db, z = DBuf(dev, x), DBuf(dev, W), DBuf(dev, np.zeros(O, np.float32)), DBuf(dev, np.zeros((B, O), np.float32))
    check(dev.h, lib().gn_dense_forward(dev.h, dx.p, dw.p, db.p, z.p, B, I, O, 6, 0))
    assert np.array_equal(_gemm(dev, 0, 1, x, W, B, O, I), z.get())


def test_gemm_split_has_no_bias(dev):
    M, N, K = 1536, 1792, 1024
    rng = np.random.default_rng(11)
    A, B = (rng.uniform(0, 1, size=s).astype(np.float32) for s in ((M, K), (N, K)))
    ref = A.astype(np.float64) @ B.astype(np.float64).T
    for sign in (np.float32(1), np.float32(-1)):
        # one downward step of half a unit per stage would be 64 * 2^-25 of the
        # mean partial sum (half of the result) = 1e-6; 1e-9 is far below one
        assert abs(np.mean((_gemm(dev, 0, 1, sign * A, B, M, N, K) - sign * ref) / ref)) <= 1e-9


def test_gemm_split_values_beyond_the_split(dev):
    """Infinities, NaN and values that round to a bf16 infinity give what IEEE
    arithmetic gives, in their tile and in no other row or column."""
    M, N, K = 1601, 1543, 128
    rng = np.random.default_rng(5)
    A, B = (rng.uniform(0.5, 1, size=s).astype(np.float32) for s in ((M, K), (N, K)))
    A[3, 7], A[200, 0], A[1600, 127], A[700, 64] = np.inf, np.nan, -np.inf, np.finfo(np.float32).max
    A[700] = np.where(np.arange(K) == 64, A[700], 0)
    B[5, 70], B[1542, 1] = np.inf, np.finfo(np.float32).max
    B[1542] *= np.float32(2.0 ** -20) * (np.arange(K) != 1) + (np.arange(K) == 1)
    with np.errstate(all="ignore"):
        ref = A.astype(np.float64) @ B.astype(np.float64).T
        ref[np.abs(ref) > np.finfo(np.float32).max] *= np.inf
    got = _gemm(dev, 0, 1, A, B, M, N, K)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[~fin & ~np.isnan(ref)], ref[~fin & ~np.isnan(ref)])
    assert np.all(np.abs(got[fin] - ref[fin]) <= 6 * K * 2.0 ** -24 * np.abs(ref[fin]))


@pytest.mark.parametrize("ta,tb", [(0, 1), (0, 0), (1, 0), (1, 1)])
def test_gemm_split_small_and_large_values(dev, ta, tb):
    """Rows of A and columns of B of any magnitude keep float32's relative
    accuracy: bf16 parts of a value near the smallest float32 must not
    underflow, nor do sums too large for the split lose their place.  Values
    are scaled per row of op(A) and column of op(B) by 2^-145 .. 2^60 (no tile
    overflows the split), in the last rows and columns by up to 2^120 (tiles
    that do, with small rows among them); sums of denormals may round at each
    of the K additions."""
    M, N, K = 1604, 1540, 448
    log(f"gemm small and large ta={ta} tb={tb}")
    rng = np.random.default_rng(ta * 2 + tb)
    ea, eb = rng.integers(-140, 61, size=(M, 1)), rng.integers(-140, 11, size=(1, N))
    ea[0], ea[1] = -145, -126
    ea[1280:], eb[:, 1280:] = rng.integers(-140, 121, size=(M - 1280, 1)), rng.integers(-140, 121, size=(1, N - 1280))
    with np.errstate(under="ignore"):
        a = np.ldexp(rng.normal(size=(M, K)), ea).astype(np.float32)
        b = np.ldexp(rng.normal(size=(K, N)), np.where(rng.random((1, N)) < 0.5, eb, 0)).astype(np.float32)
    got = _gemm(dev, ta, tb, np.ascontiguousarray(a.T) if ta else a, np.ascontiguousarray(b.T) if tb else b, M, N, K)
    a, b = a.astype(np.float64), b.astype(np.float64)
    ref, mag = a @ b, np.abs(a) @ np.abs(b)
    fin = mag < np.finfo(np.float32).max  # no partial sum overflows
    assert np.isfinite(got[fin]).all()
    assert np.all(np.abs(got[fin] - ref[fin]) <= 6 * K * 2.0 ** -24 * mag[fin] + K * 2.0 ** -149)
    tiny = fin & (mag < 2.0 ** -80) & (mag > 2.0 ** -100)
    assert tiny.any()
    err = (got[tiny] - ref[tiny]) / mag[tiny]
    assert np.sqrt(np.mean(err * err)) <= 2.0 ** -24  # as for ordinary values: test_gemm_split's norm bound over sqrt(K)


def test_forward_products_keep_their_order_of_fp32_sums(dev):
    """A forward product without bias (SwiGLU's [W x | V x]) has the bits of a
    linear Dense layer of the same sizes with zero biases, in 128-wide tiles too."""
    from goneuron_amd._lib import check, lib
    B, I, O = 1604, 512, 800  # 13 x 13 tiles of 128
    log("swiglu forward product")
    rng = np.random.default_rng(3)
    x, W = rng.normal(size=(B, I)).astype(np.float32), rng.normal(size=(2 * O, I)).astype(np.float32)
    dx, dw, db = DBuf(dev, x), DBuf(dev, W), DBuf(dev, np.zeros(2 * O, np.float32))
    z, out, work = (DBuf(dev, np.zeros(s, np.float32)) for s in ((B, 2 * O), (B, O), (4 * B, O)))
    check(dev.h, lib().gn_dense_forward(dev.h, dx.p, dw.p, db.p, z.p, B, I, 2 * O, 6, 0))
    check(dev.h, lib().gn_swiglu_forward(dev.h, dx.p, dw.p, out.p, work.p, B, I, O))
    assert np.array_equal(work.get()[:2 * B].reshape(B, 2 * O), z.get())
