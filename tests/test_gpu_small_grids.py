"""Small grids, whose K is dealt to groups of waves inside a workgroup (and,
for a long K, to chunks): sizes around the 32- and 64-wide tiles, K around the
16-deep steps and the 4, 8 and 16 groups (fewer steps than groups, one more,
a remainder in the last), and grids on both sides of every bound of the
choice.  Against the oracle's bound; repeated calls give the same bits; beta
== 0 does not read C; the bias and activation come after the groups' sum."""
import zlib

import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc
from tests.helpers import Case

pytestmark = pytest.mark.gpu

MODES = [ug.MODE_FP32, ug.MODE_FP32_MFMA, ug.MODE_DGEMM]
# One tile; up to 256, 512 tiles of 32x32; up to 256, 512 of 64x64; more.
GRIDS = [(1, 1), (31, 33), (65, 64), (512, 511), (513, 512), (700, 720), (1023, 1023), (1025, 1000), (1410, 1400),
         (1500, 1500)]
KS = [1, 15, 16, 17, 65, 127, 129, 257, 300]
LONG = [(33, 40, 2100), (64, 64, 5000), (500, 500, 4200), (640, 520, 4100), (100, 90, 1300), (1100, 300, 2600)]


def device_product(mode, case, c0):
    dA, dB, dC = hip.DeviceArray.from_host(case.A), hip.DeviceArray.from_host(case.B), hip.DeviceArray.from_host(c0)
    fn = ug.dgemm_dev if mode == ug.MODE_DGEMM else ug.sgemm_dev
    kw = {} if mode == ug.MODE_DGEMM else {"mode": mode}
    fn(case.major, case.ta, case.tb, case.M, case.N, case.K, case.alpha, dA, case.lda, dB, case.ldb, case.beta, dC,
       case.ldc, **kw)
    hip.synchronize()
    out = dC.download()
    for d in (dA, dB, dC):
        d.free()
    return out


def check(mode, ta, tb, M, N, K, beta):
    double = mode == ug.MODE_DGEMM
    case = Case("R", ta, tb, M, N, K, 1.5, beta, seed=zlib.crc32(f"small{mode}{ta}{tb}{M},{N},{K}".encode()),
                dtype=np.float64 if double else np.float32)
    c0 = case.C0 if beta else np.full_like(case.C0, np.nan)
    print(f"mode {mode} {ta}{tb} {M}x{N}x{K} beta {beta}", flush=True)
    got = device_product(mode, case, c0)
    assert got.tobytes() == device_product(mode, case, c0).tobytes(), f"{M}x{N}x{K}: not repeatable"
    ok, worst = case.judge(got, eps=orc.EPS64 if double else orc.EPS32)
    assert ok, f"{M}x{N}x{K}: worst/bound {worst:.3g}"


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_group_and_tile_edges(mode, ta, tb):
    for i, (M, N) in enumerate(GRIDS):
        for K in (KS if M < 600 else KS[i % 3::3]):
            check(mode, ta, tb, M, N, K, 0.5 if (i + K) % 2 else 0.0)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "T")])
def test_long_k_on_small_grids(mode, ta, tb):
    for M, N, K in LONG:
        check(mode, ta, tb, M, N, K, 0.5)


@pytest.mark.parametrize("mode", [ug.MODE_FP32, ug.MODE_FP32_MFMA])
@pytest.mark.parametrize("M,N,K", [(40, 50, 200), (600, 650, 90), (1000, 900, 130), (64, 40, 5000)])
def test_epilogue_after_the_groups_sum(mode, M, N, K):
    g = orc.rng(M + N + K + mode)
    A, B, C0, bias = orc.uniform(g, (M, K)), orc.uniform(g, (K, N)), orc.uniform(g, (M, N)), orc.uniform(g, (N,))
    dA, dB, dC, db = (hip.DeviceArray.from_host(x) for x in (A, B, C0, bias))
    ug.sgemm_ex_dev("R", "N", "N", M, N, K, 1.25, dA, K, dB, N, 0.5, dC, N, mode=mode, bias=db, bias_dim=ug.BIAS_COLS,
                    act=ug.ACT_LEAKY_RELU, slope=0.1)
    hip.synchronize()
    pre = 1.25 * (A.astype(np.float64) @ B.astype(np.float64)) + 0.5 * C0 + bias[None, :]
    want = np.where(pre > 0, pre, np.float64(np.float32(0.1)) * pre)
    scale = 1.25 * (np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)) + 0.5 * np.abs(C0) + np.abs(bias)
    got = dC.download().astype(np.float64)
    assert np.all(np.abs(got - want) <= orc.tolerance(K + 2) * scale)


@pytest.mark.parametrize("mode", [ug.MODE_FP32, ug.MODE_FP32_MFMA])
@pytest.mark.parametrize("M,N,K", [(1984, 2048, 4096), (1000, 1024, 16384), (1400, 1400, 30000)])
def test_partial_sums_fit_the_static_scratch(mode, M, N, K):
    """The no-allocation entry takes these sizes: few enough tiles to split K,
    but with chunks of it whose partial sums could pass 64 MiB."""
    dA, dB = hip.DeviceArray((M, K), np.float32), hip.DeviceArray((K, N), np.float32)
    for d in (dA, dB):
        hip.check(hip.lib().hipMemset(d.ptr, 0, d.nbytes), "clear")
    dC = hip.DeviceArray.from_host(np.ones((M, N), np.float32))
    ug.sgemm_noalloc_dev("R", "N", "N", M, N, K, 1.0, dA, K, dB, N, 0.5, dC, N, mode=mode)
    hip.synchronize()
    assert np.all(dC.download() == 0.5)
