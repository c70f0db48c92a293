"""Operands at any element alignment and every remainder of a tile, row or
16-byte load: the same product from packed, aligned operands and from operands
that start 1-3 elements off, have odd leading dimensions and lie between NaNs
(before, after and in the gaps between rows) gives the same bits, and C's own
gaps keep their values.  The packed result is held to the oracle's bound."""
import zlib

import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc
from tests.helpers import Case, MODE_EXTRA

pytestmark = pytest.mark.gpu

# Rows shorter than one 16-byte load, one element around loads, k slabs and
# tiles, and sides of several tiles that end one element early or late.
SHAPES = [(1, 1, 1), (3, 2, 3), (2, 5, 4), (5, 67, 3), (65, 2, 19), (67, 66, 63), (130, 71, 33), (129, 255, 130),
          (259, 130, 17), (31, 33, 515)]


def guarded(x, rows, length, off, pad):
    """(device buffer, element offset, ld) of rows x length inside NaNs."""
    ld = length + pad
    h = np.full(off + rows * ld + 8, np.nan, x.dtype)
    h[off:off + rows * ld].reshape(rows, ld)[:, :length] = x
    return hip.DeviceArray.from_host(h), off, ld


def product(mode, case, off, pad, double):
    """C (logical) and whether everything around it kept its values."""
    row_a, row_b = case.lda, case.ldb   # packed cases: ld is the row length
    bufs = [guarded(x, x.shape[0], n, o, p) for x, n, o, p in
            ((case.A, row_a, off, pad), (case.B, row_b, (off + 1) % 4 if off else 0, pad and pad + 2),
             (case.C0, case.ldc, (off + 2) % 4 if off else 0, pad))]
    (dA, oa, lda), (dB, ob, ldb), (dC, oc, ldc) = bufs
    fn = ug.dgemm_dev if double else ug.sgemm_dev
    kw = {} if double else {"mode": mode}
    fn(case.major, case.ta, case.tb, case.M, case.N, case.K, case.alpha, dA.at(oa), lda, dB.at(ob), ldb, case.beta,
       dC.at(oc), ldc, **kw)
    hip.synchronize()
    h = dC.download()
    rows = case.C0.shape[0]
    body = h[oc:oc + rows * ldc].reshape(rows, ldc)
    around = np.concatenate([h[:oc], h[oc + rows * ldc:], body[:, case.ldc:].ravel()])
    for d in (dA, dB, dC):
        d.free()
    return np.ascontiguousarray(body[:, :case.ldc]), bool(np.all(np.isnan(around)))


@pytest.mark.parametrize("mode", [ug.MODE_FP32, ug.MODE_FP32_MFMA, ug.MODE_DGEMM, ug.MODE_BF16X3, ug.MODE_FP16X3,
                                  ug.MODE_BF16X1, ug.MODE_BF16X6, ug.MODE_FP8_BLOCK])
@pytest.mark.parametrize("major,ta,tb", [("R", "N", "N"), ("R", "N", "T"), ("R", "T", "N"), ("R", "T", "T"),
                                         ("C", "N", "N"), ("C", "T", "N")])
def test_unaligned_operands_give_the_packed_bits(mode, major, ta, tb):
    double = mode == ug.MODE_DGEMM
    for (M, N, K) in SHAPES:
        case = Case(major, ta, tb, M, N, K, 1.5, 0.5, seed=zlib.crc32(f"edge{mode}{major}{ta}{tb}{M},{N},{K}".encode()),
                    dtype=np.float64 if double else np.float32)
        print(f"mode {mode} {major}{ta}{tb} {M}x{N}x{K}", flush=True)
        packed, kept = product(mode, case, 0, 0, double)
        assert kept
        if mode != ug.MODE_FP8_BLOCK:
            exact, scale = case.exact()
            tol = orc.tolerance(K, eps=orc.EPS64 if double else orc.EPS32, extra=MODE_EXTRA.get(mode, 0.0))
            ok, worst = orc.check_bound(case.logical(packed), exact, scale, tol)
            assert ok, f"{M}x{N}x{K}: worst/bound {worst:.3g}"
        for off, pad in ((1, 1), (3, 6)):
            got, kept = product(mode, case, off, pad, double)
            assert kept, f"{M}x{N}x{K} offset {off}: wrote outside C"
            assert got.tobytes() == packed.tobytes(), f"{M}x{N}x{K} offset {off} pad {pad}: bits differ"
