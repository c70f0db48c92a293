"""Automatic tile shapes of grids beyond one 128x128 tile a CU, where the tiles
of the fullest CU decide: sizes on both sides of whole rounds and long, flat
ones, with ragged edges, a short and an odd K, padded rows, every layout, C
read and not.  Against the oracle's bound; repeated calls give the same bits."""
import zlib

import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc
from tests.helpers import Case

pytestmark = pytest.mark.gpu

SIZES = [(2050, 2049, 33), (2111, 2177, 67), (770, 5500, 130), (6662, 808, 50), (3000, 2900, 17), (4097, 2111, 40)]


@pytest.mark.parametrize("mode", [ug.MODE_FP32, ug.MODE_FP32_MFMA])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_tile_choice(mode, ta, tb):
    for i, (M, N, K) in enumerate(SIZES):
        beta = 0.5 if i % 2 else 0.0
        case = Case("R", ta, tb, M, N, K, 1.5, beta, seed=zlib.crc32(f"tc{mode}{ta}{tb}{M}".encode()), pad=i % 3)
        c0 = case.C0 if beta else np.full_like(case.C0, np.nan)
        dA, dB = hip.DeviceArray.from_host(case.A), hip.DeviceArray.from_host(case.B)
        got = []
        print(f"mode {mode} {ta}{tb} {M}x{N}x{K}", flush=True)
        for _ in range(2):
            dC = hip.DeviceArray.from_host(c0)
            ug.sgemm_dev("R", ta, tb, M, N, K, 1.5, dA, case.lda, dB, case.ldb, beta, dC, case.ldc, mode=mode)
            hip.synchronize()
            got.append(dC.download())
            dC.free()
        dA.free()
        dB.free()
        assert got[0].tobytes() == got[1].tobytes()
        Aop = (case.A[:, :M].T if ta == "T" else case.A[:, :K]).astype(np.float64)
        Bop = (case.B[:, :K].T if tb == "T" else case.B[:, :N]).astype(np.float64)
        scale = 1.5 * (np.abs(Aop) @ np.abs(Bop)) + beta * np.abs(case.C0[:, :N])
        want = 1.5 * (Aop @ Bop) + beta * case.C0[:, :N]
        ok, worst = orc.check_bound(got[0][:, :N], want, scale, orc.tolerance(K + 2))
        assert ok, f"{M}x{N}x{K}: {worst:.3g}"
        assert np.array_equal(got[0][:, N:], c0[:, N:], equal_nan=True)


@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_tile_choice_fp64(ta, tb):
    for M, N, K in [(2050, 2049, 33), (770, 5500, 50), (6240, 808, 40)]:
        case = Case("R", ta, tb, M, N, K, 1.5, 0.5, seed=M, dtype=np.float64, pad=1)
        dA, dB, dC = (hip.DeviceArray.from_host(x) for x in (case.A, case.B, case.C0))
        print(f"fp64 {ta}{tb} {M}x{N}x{K}", flush=True)
        ug.dgemm_dev("R", ta, tb, M, N, K, 1.5, dA, case.lda, dB, case.ldb, 0.5, dC, case.ldc)
        hip.synchronize()
        got = dC.download()
        for d in (dA, dB, dC):
            d.free()
        Aop = case.A[:, :M].T if ta == "T" else case.A[:, :K]
        Bop = case.B[:, :K].T if tb == "T" else case.B[:, :N]
        want = 1.5 * (Aop @ Bop) + 0.5 * case.C0[:, :N]
        scale = 1.5 * (np.abs(Aop) @ np.abs(Bop)) + 0.5 * np.abs(case.C0[:, :N])
        # Both sides are FP64 sums of K products: twice the bound of one.
        assert np.all(np.abs(got[:, :N] - want) <= 2 * (K + 4) * np.finfo(np.float64).eps * scale)
        assert np.array_equal(got[:, N:], case.C0[:, N:])


@pytest.mark.parametrize("mode", [ug.MODE_BF16X1, ug.MODE_BF16X3, ug.MODE_FP16X3])
def test_large_tiles_a_little_over(mode):
    """17 x 16 tiles of 256x256: the automatic choice and the large tile give the same bits."""
    M, N, K = 4200, 4090, 70
    case = Case("R", "N", "T", M, N, K, 1.0, 0.0, seed=mode)
    dA, dB = hip.DeviceArray.from_host(case.A), hip.DeviceArray.from_host(case.B)
    got = []
    for variant in (-1, 6):
        ug.force_variant(mode, variant)
        dC = hip.DeviceArray.from_host(np.full((M, N), np.nan, np.float32))
        ug.sgemm_dev("R", "N", "T", M, N, K, 1.0, dA, K, dB, K, 0.0, dC, N, mode=mode)
        hip.synchronize()
        got.append(dC.download())
        dC.free()
    ug.force_variant(mode, -1)
    dA.free()
    dB.free()
    assert got[0].tobytes() == got[1].tobytes()
