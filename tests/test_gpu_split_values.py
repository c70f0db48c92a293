"""The split of infinities, NaNs, values that round up to infinity and
subnormals, wherever it runs: in a preparation pass, in a core that splits an
operand while staging it (tiles inside and at the edge, an odd last row, a
ragged last K step) and in the small-grid kernel.  Where a result is finite,
infinite (and its sign) or NaN follows from the planes alone, whatever the
order of the sum; rows without such values stay within the oracle's bound."""
import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc
from tests.helpers import MODE_EXTRA

pytestmark = pytest.mark.gpu

NP = {ug.MODE_BF16X1: 1, ug.MODE_BF16X3: 2, ug.MODE_BF16X6: 3, ug.MODE_FP16X3: 2}
PAIRS = {1: [(0, 0)], 2: [(1, 0), (0, 1), (0, 0)], 3: [(2, 0), (0, 2), (1, 1), (1, 0), (0, 1), (0, 0)]}


def bf16(x):
    u = np.ascontiguousarray(x, np.float32).view(np.uint32).astype(np.uint64)
    r = ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).astype(np.uint32).view(np.float32)
    return np.where(np.isnan(x), x, r)


def planes(mode, X):
    """Planes of X (rows of op(A) or columns of op(B) as rows), as float64."""
    rnd = bf16
    if mode == ug.MODE_FP16X3:
        amax = np.nanmax(np.abs(X), axis=1)
        e = np.where(np.isfinite(amax) & (amax > 0), np.frexp(amax)[1], 0) - 15
        X = np.ldexp(X, -e[:, None]).astype(np.float32)
        rnd = lambda v: v.astype(np.float16).astype(np.float32)
    out = [rnd(X)]
    for p in range(1, NP[mode]):
        X = np.where(np.isfinite(out[-1]), X - out[-1], np.float32(0)) if p == 1 else X - out[-1]
        out.append(rnd(X))
    return [o.astype(np.float64) for o in out]


@pytest.mark.parametrize("mode", list(NP))
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_special_values(mode, ta, tb):
    g = orc.rng(17)
    for M, N, K in [(71, 301, 100), (301, 71, 100), (1, 65, 70), (513, 130, 1100)]:
        A = orc.uniform(g, (M, K)).astype(np.float32)
        B = orc.uniform(g, (N, K)).astype(np.float32)
        special = [np.inf, -np.inf, np.nan, 3.4e38, -3.3961776e38, 1e-40]
        rows = [r for r in (0, 5, 17, 40, 66, 70) if r < M]
        for i, r in enumerate(rows if M > 1 else []):
            A[r, (r * 7 + 3) % K] = special[i]
        cols = [c for c in (2, 64, N - 1) if c < N]
        for i, c in enumerate(cols):
            B[c, K - 1 - i] = special[i]
        with np.errstate(all="ignore"):
            pa, pb = planes(mode, A), planes(mode, B)
            want = sum(pa[i] @ pb[j].T for i, j in PAIRS[NP[mode]])
            exact = A.astype(np.float64) @ B.astype(np.float64).T
            scale = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64).T
        # A large finite magnitude overflows nothing but its own planes.
        plain = np.ix_([r for r in range(M) if np.all(np.abs(A[r]) <= 1)], [c for c in range(N) if np.all(np.abs(B[c]) <= 1)])
        a, b = (A.T if ta == "T" else A), (B if tb == "T" else B.T)
        dA, dB = hip.DeviceArray.from_host(np.ascontiguousarray(a)), hip.DeviceArray.from_host(np.ascontiguousarray(b))
        try:
            for variant, splits in [(-1, 0), (3, 1), (7, 1), (4, 1), (6, 2)]:
                ug.force_variant(mode, variant)
                ug.force_splits(mode, splits)
                print(f"mode {mode} {ta}{tb} {M}x{N}x{K} variant {variant}", flush=True)
                dC = hip.DeviceArray.from_host(np.zeros((M, N), np.float32))
                ug.sgemm_dev("R", ta, tb, M, N, K, 1.0, dA, a.shape[1], dB, b.shape[1], 0.0, dC, N, mode=mode)
                hip.synchronize()
                got = dC.download()
                dC.free()
                bad = ~np.isfinite(want)
                assert np.array_equal(np.isnan(got[bad]), np.isnan(want[bad]))
                inf = np.isinf(want)
                assert np.array_equal(got[inf], want[inf].astype(np.float32))
                ok, worst = orc.check_bound(got[plain], exact[plain], scale[plain],
                                            orc.tolerance(K + 2, extra=MODE_EXTRA[mode]))
                assert ok, worst
        finally:
            ug.force_variant(mode, -1)
            ug.force_splits(mode, 0)
            dA.free()
            dB.free()


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("K", [64, 65, 200, 300, 513, 1100, 2048, 2049, 8192, 8200])
def test_row_scales(K, ta, tb):
    """FP16X3's preparation: pairs of whole rows on 16 .. 256 threads, maxima
    in parts and combined, columns by 64 and by 256, with and without an operand
    that the core splits; wide data, so that a wrong scale shows."""
    mode = ug.MODE_FP16X3
    g = orc.rng(K)
    for M, N in [(70, 333), (600, 130)] + ([(64, 20000)] if K in (200, 2049) else []):
        A, B = orc.wide_range(g, (M, K)).astype(np.float32), orc.wide_range(g, (N, K)).astype(np.float32)
        a, b = np.ascontiguousarray(A.T if ta == "T" else A), np.ascontiguousarray(B if tb == "T" else B.T)
        exact = A.astype(np.float64) @ B.astype(np.float64).T
        scale = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64).T
        dA, dB = hip.DeviceArray.from_host(a), hip.DeviceArray.from_host(b)
        try:
            for variant in (3, 7):
                ug.force_variant(mode, variant)
                ug.force_splits(mode, 1)
                print(f"K {K} {ta}{tb} {M}x{N} variant {variant}", flush=True)
                dC = hip.DeviceArray.from_host(np.zeros((M, N), np.float32))
                ug.sgemm_dev("R", ta, tb, M, N, K, 1.0, dA, a.shape[1], dB, b.shape[1], 0.0, dC, N, mode=mode)
                hip.synchronize()
                got = dC.download()
                dC.free()
                ok, worst = orc.check_bound(got, exact, scale, orc.tolerance(K + 2, extra=MODE_EXTRA[mode]))
                assert ok, worst
        finally:
            ug.force_variant(mode, -1)
            ug.force_splits(mode, 0)
            dA.free()
            dB.free()
