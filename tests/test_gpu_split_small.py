"""Split forms on small grids, one launch without planes: sizes around the 32-
and 64-wide tiles and the bounds of the choice, K around the 32-deep steps
and the 8 and 16 waves of a workgroup, every layout, odd leading dimensions
between NaNs, epilogue and beta == 0.  FP16X3 against the exact emulation of
its split (wide data: the row scales matter), the BF16 forms against theirs;
every form against the oracle's bound.  Repeated calls give the same bits, and
the no-allocation entry the same as the other."""
import zlib

import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc
from tests.helpers import Case, MODE_EXTRA

pytestmark = pytest.mark.gpu

MODES = {ug.MODE_BF16X1: 1, ug.MODE_BF16X3: 2, ug.MODE_BF16X6: 3, ug.MODE_FP16X3: 0}   # planes (0: fp16)
SHAPES = [(1, 1, 1), (3, 33, 7), (31, 32, 8), (33, 65, 31), (64, 15, 32), (65, 100, 33), (17, 40, 511), (40, 70, 513),
          (100, 90, 1100), (512, 512, 40), (513, 512, 100), (64, 33, 2048), (30, 31, 3072), (1024, 1000, 96),
          (1025, 1024, 64), (1400, 1330, 256), (2048, 2000, 64)]


def emulation(mode, A, B):
    return orc.fp16x3_product(A, B) if mode == ug.MODE_FP16X3 else orc.bf16_product(A, B, MODES[mode])


def run(mode, case, dA, dB, c0, entry):
    dC = hip.DeviceArray.from_host(c0)
    entry("R", case.ta, case.tb, case.M, case.N, case.K, case.alpha, dA, case.lda, dB, case.ldb, case.beta, dC,
          case.ldc, mode=mode)
    hip.synchronize()
    out = dC.download()
    dC.free()
    return out


@pytest.mark.parametrize("mode", list(MODES))
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_small_grids(mode, ta, tb):
    for i, (M, N, K) in enumerate(SHAPES):
        beta = 0.5 if i % 2 else 0.0
        case = Case("R", ta, tb, M, N, K, 1.5, beta, seed=zlib.crc32(f"ss{mode}{ta}{tb}{M},{N},{K}".encode()),
                    dist="wide" if i % 3 == 2 else "uniform", pad=i % 4)
        # Nothing outside the operands is read into the result: NaN in the gaps between rows.
        for X, n in ((case.A, M if ta == "T" else K), (case.B, K if tb == "T" else N)):
            X[:, n:] = np.nan
        dA, dB = hip.DeviceArray.from_host(case.A), hip.DeviceArray.from_host(case.B)
        c0 = case.C0 if beta else np.full_like(case.C0, np.nan)
        print(f"mode {mode} {ta}{tb} {M}x{N}x{K} pad {i % 4}", flush=True)
        got = run(mode, case, dA, dB, c0, ug.sgemm_dev)
        assert got.tobytes() == run(mode, case, dA, dB, c0, ug.sgemm_dev).tobytes()
        assert got.tobytes() == run(mode, case, dA, dB, c0, ug.sgemm_noalloc_dev).tobytes()
        Aop = (case.A[:, :M].T if ta == "T" else case.A[:, :K]).astype(np.float32)
        Bop = (case.B[:, :K].T if tb == "T" else case.B[:, :N]).astype(np.float32)
        scale = 1.5 * (np.abs(Aop).astype(np.float64) @ np.abs(Bop).astype(np.float64)) + beta * np.abs(case.C0[:, :N])
        if M * N * K <= 4e6:
            want = 1.5 * emulation(mode, np.ascontiguousarray(Aop), np.ascontiguousarray(Bop)) + beta * case.C0[:, :N]
            ok, worst = orc.check_bound(got[:, :N], want, scale, orc.tolerance(K + 2))
            assert ok, f"{M}x{N}x{K} against the emulation: {worst:.3g}"
        want = 1.5 * (Aop.astype(np.float64) @ Bop.astype(np.float64)) + beta * case.C0[:, :N]
        ok, worst = orc.check_bound(got[:, :N], want, scale, orc.tolerance(K + 2, extra=MODE_EXTRA[mode]))
        assert ok, f"{M}x{N}x{K}: {worst:.3g}"
        assert np.array_equal(got[:, N:], c0[:, N:], equal_nan=True)


@pytest.mark.parametrize("mode", [ug.MODE_BF16X3, ug.MODE_FP16X3])
@pytest.mark.parametrize("M,N,K,bias_dim", [(40, 50, 200, ug.BIAS_ROWS), (600, 650, 90, ug.BIAS_COLS),
                                           (1000, 1000, 130, ug.BIAS_ROWS)])
def test_epilogue(mode, M, N, K, bias_dim):
    g = orc.rng(M + N + K + mode)
    A, B, C0 = orc.uniform(g, (M, K)), orc.uniform(g, (K, N)), orc.uniform(g, (M, N))
    bias = orc.uniform(g, (M if bias_dim == ug.BIAS_ROWS else N,))
    dA, dB, dC, db = (hip.DeviceArray.from_host(x) for x in (A, B, C0, bias))
    ug.sgemm_ex_dev("R", "N", "N", M, N, K, 1.25, dA, K, dB, N, 0.5, dC, N, mode=mode, bias=db, bias_dim=bias_dim,
                    act=ug.ACT_LEAKY_RELU, slope=0.1)
    hip.synchronize()
    b = bias[:, None] if bias_dim == ug.BIAS_ROWS else bias[None, :]
    pre = 1.25 * (A.astype(np.float64) @ B.astype(np.float64)) + 0.5 * C0 + b
    want = np.where(pre > 0, pre, np.float64(np.float32(0.1)) * pre)
    scale = 1.25 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)) + 0.5 * np.abs(C0) + np.abs(b)
    got = dC.download().astype(np.float64)
    assert np.all(np.abs(got - want) <= orc.tolerance(K + 2, extra=MODE_EXTRA[mode]) * scale)


@pytest.mark.parametrize("mode", list(MODES))
def test_rows_of_zeros_infinities_and_nan(mode):
    """A zero row, a row with an infinity and one with a NaN: the first gives
    zeros, the others nothing finite, and their neighbours are untouched."""
    M, N, K = 70, 40, 96
    A, B = np.ones((M, K), np.float32), np.ones((K, N), np.float32)
    A[3], A[5, 7], A[9, 90] = 0.0, np.inf, np.nan
    C = np.zeros((M, N), np.float32)
    ug.sgemm("R", "N", "N", M, N, K, 1.0, A, K, B, N, 0.0, C, N, mode=mode)
    assert np.all(C[3] == 0.0) and not np.any(np.isfinite(C[[5, 9]]))
    assert np.all(C[np.setdiff1d(np.arange(M), [3, 5, 9])] == K)
