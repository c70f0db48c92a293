"""Split forms on grids smaller than the chip: the automatic choice of tile and
split count, at sides around its 64-, 128- and 256-wide tiles and K that
divides into whole and ragged chunks, every layout, odd pitches, against the
oracle's bound; the no-allocation entry chooses alike, runs what the choice by
the grid alone runs there, and refuses what that is refused."""
import zlib

import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc
from tests.helpers import Case, MODE_EXTRA

pytestmark = pytest.mark.gpu

MODES = [ug.MODE_BF16X1, ug.MODE_BF16X3, ug.MODE_BF16X6, ug.MODE_FP16X3]
SHAPES = [(493, 700, 4099), (64, 1500, 3300), (1500, 35, 4500), (257, 513, 6000), (1030, 1025, 2080), (127, 862, 5001)]


def call(entry, mode, case, dA, dB):
    dC = hip.DeviceArray.from_host(case.C0)
    try:
        entry("R", case.ta, case.tb, case.M, case.N, case.K, case.alpha, dA, case.lda, dB, case.ldb, case.beta, dC,
              case.ldc, mode=mode)
        hip.synchronize()
        return dC.download()
    finally:
        dC.free()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
def test_choice(mode, ta, tb):
    for i, (M, N, K) in enumerate(SHAPES):
        case = Case("R", ta, tb, M, N, K, 1.5, 0.5, seed=zlib.crc32(f"sp{mode}{ta}{tb}{M}".encode()), pad=i % 3)
        dA, dB = hip.DeviceArray.from_host(case.A), hip.DeviceArray.from_host(case.B)
        print(f"mode {mode} {ta}{tb} {M}x{N}x{K}", flush=True)
        got = call(ug.sgemm_dev, mode, case, dA, dB)
        assert got.tobytes() == call(ug.sgemm_dev, mode, case, dA, dB).tobytes()
        assert got.tobytes() == call(ug.sgemm_noalloc_dev, mode, case, dA, dB).tobytes()
        Aop = (case.A[:, :M].T if ta == "T" else case.A[:, :K]).astype(np.float64)
        Bop = (case.B[:, :K].T if tb == "T" else case.B[:, :N]).astype(np.float64)
        scale = 1.5 * (np.abs(Aop) @ np.abs(Bop)) + 0.5 * np.abs(case.C0[:, :N])
        ok, worst = orc.check_bound(got[:, :N], 1.5 * (Aop @ Bop) + 0.5 * case.C0[:, :N], scale,
                                    orc.tolerance(K + 2, extra=MODE_EXTRA[mode]))
        assert ok, f"{M}x{N}x{K}: {worst:.3g}"
        dA.free()
        dB.free()


@pytest.mark.parametrize("M,N,K,fits", [(493, 2304, 5000, True), (64, 6272, 6592, False), (1, 12000, 2048, False)])
def test_no_allocation_limits(M, N, K, fits):
    """BF16X3.  493x2304x5000: planes of 57 MB, with the partial sums of the
    fastest split count more than the scratch.  64x6272x6592 (167 MB of planes)
    and 1x12000x2048 (99 MB) need less than that by other routes."""
    case = Case("R", "N", "N", M, N, K, 1.0, 0.0, seed=K)
    dA, dB = hip.DeviceArray.from_host(case.A), hip.DeviceArray.from_host(case.B)
    want = call(ug.sgemm_dev, ug.MODE_BF16X3, case, dA, dB)
    if fits:
        assert want.tobytes() == call(ug.sgemm_noalloc_dev, ug.MODE_BF16X3, case, dA, dB).tobytes()
    else:
        with pytest.raises(ug.UgemmError) as e:
            call(ug.sgemm_noalloc_dev, ug.MODE_BF16X3, case, dA, dB)
        assert e.value.status == ug.ERR_SCRATCH
