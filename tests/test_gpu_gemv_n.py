"""gemv 'N' over its three ways: one thread a row, 16 waves to 64 rows in one
launch, and in chunks of columns; rows around 64, columns around 128, the
bounds of the choice and ragged chunks; strides, a padded leading dimension,
beta == 0 not reading y.  Against FP64 sums (numpy.longdouble for FP64), bound
by the length of the sum; repeated calls give the same bits."""
import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SIZES = [(1, 1), (1, 128), (63, 127), (64, 128), (65, 129), (300, 768), (130, 769), (1000, 1024), (200, 1025),
         (70, 1300), (3, 20000), (192, 17216), (4097, 333), (33000, 130), (4095, 2000), (16500, 4100)]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("beta,incx,incy,pad", [(0.0, 1, 1, 0), (0.5, 2, 3, 5)])
def test_gemv_n(dtype, beta, incx, incy, pad):
    wide = np.float64 if dtype == np.float32 else np.longdouble
    eps = np.finfo(dtype).eps
    for M, N in SIZES:
        if M * N > 2e7 and (pad or dtype == np.float32):
            continue
        g = orc.rng(M + N)
        A = orc.uniform(g, (N, M + pad)).astype(dtype)
        A[:, M:] = np.nan
        x = np.full(N * incx, np.nan, dtype)
        x[::incx] = orc.uniform(g, (N,)).astype(dtype)
        y0 = np.full(M * incy, np.nan, dtype)
        if beta:
            y0[::incy] = orc.uniform(g, (M,)).astype(dtype)
        dA, dx = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(x)
        got = []
        print(f"{np.dtype(dtype).name} {M}x{N} beta {beta}", flush=True)
        for _ in range(2):
            dy = hip.DeviceArray.from_host(y0)
            ug.gemv_dev("N", M, N, 1.5, dA, M + pad, dx, incx, beta, dy, incy, double=dtype == np.float64)
            hip.synchronize()
            got.append(dy.download())
            dy.free()
        dA.free()
        dx.free()
        assert got[0].tobytes() == got[1].tobytes()
        a, xs = A[:, :M], x[::incx]
        want = 1.5 * (xs.astype(wide) @ a.astype(wide))
        bound = 1.5 * (np.abs(xs).astype(wide) @ np.abs(a).astype(wide))
        if beta:
            want = want + beta * y0[::incy].astype(wide)
            bound = bound + beta * np.abs(y0[::incy])
        assert np.all(np.abs(got[0][::incy] - want) <= (N + 4) * eps * bound)
        if incy > 1:
            assert np.all(np.isnan(np.delete(got[0], np.s_[::incy])))


def test_gemv_n_of_nearly_2_to_the_31_columns():
    """Chunk bounds beyond INT_MAX: one row of 2^31 - 100 ones (17 GB with x).
    The blocks' sums are exact; at most 32 roundings follow, each by half a
    step of the total (64) or less."""
    N = 2 ** 31 - 100
    ones, block = [hip.DeviceArray(N, np.float32) for _ in range(2)], np.ones(1 << 24, np.float32)
    for d in ones:
        hip.check(hip.lib().hipMemcpy(d.ptr, block.ctypes.data, block.nbytes, hip.H2D), "fill")
        for at in range(block.size, N, block.size):
            hip.check(hip.lib().hipMemcpy(d.at(at), d.ptr, 4 * min(block.size, N - at), hip.D2D), "fill")
    dy = hip.DeviceArray(1, np.float32)
    ug.gemv_dev("N", 1, N, 1.0, ones[0], 1, ones[1], 1, 0.0, dy, 1)
    hip.synchronize()
    got = float(dy.download()[0])
    for d in ones:
        d.free()
    assert abs(got - N) <= 32 * 64, got


def plain_sums(A, x, chunk=64):
    """A^T x by one thread a row: chunks of columns on four accumulators (one
    rounding a multiply-add), the chunks' sums one after the other."""
    wide = np.float64 if A.dtype == np.float32 else np.longdouble
    y = np.zeros(A.shape[1], A.dtype)
    for c in range(0, len(x), chunk):
        s = [np.zeros_like(y) for _ in range(4)]
        for n in range(c, min(c + chunk, len(x))):
            i = (n - c) % 4
            s[i] = (A[n].astype(wide) * wide(x[n]) + s[i]).astype(A.dtype)
        y = y + ((s[0] + s[1]) + (s[2] + s[3]))
    return y


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_gemv_n_sums_of_few_columns_are_no_less_exact(dtype):
    """The waves' sums are added in pairs: the root mean square error over rows
    of 128 to 250 columns stays below that of a thread's own sums."""
    wide = np.float64 if dtype == np.float32 else np.longdouble
    got = want = 0.0
    for N in (128, 160, 200, 250):
        for seed in range(5):
            g = np.random.default_rng(1000 * N + seed)
            A, x = g.standard_normal((N, 400)).astype(dtype), g.standard_normal(N).astype(dtype)
            exact = x.astype(wide) @ A.astype(wide)
            dA, dx, dy = hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(x), hip.DeviceArray(400, dtype)
            ug.gemv_dev("N", 400, N, 1.0, dA, 400, dx, 1, 0.0, dy, 1, double=dtype == np.float64)
            hip.synchronize()
            # Relative to sqrt(N), which the errors of both grow with.
            got += float(np.sum((dy.download() - exact) ** 2)) / N
            want += float(np.sum((plain_sums(A, x) - exact) ** 2)) / N
    print(f"{np.dtype(dtype).name}: {np.sqrt(got / want):.3f} of the plain sums' error")
    assert got <= want
