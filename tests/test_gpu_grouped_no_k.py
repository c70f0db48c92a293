"""Grouped split-form plans with problems that have nothing to multiply (K == 0
or alpha == 0, whose A and B may be NULL): they come out as beta * C exactly
and read neither operand, beside ordinary problems that meet their
form's bound.  Both layouts of B, the variants that split B in the core, and
the default."""
import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from tests.helpers import Case

pytestmark = pytest.mark.gpu

# Sizes at one row or column, within and past the tiles of 64 and 128.
EMPTY = [(1, 1, 0, 1.0), (33, 17, 0, 1.5), (40, 50, 60, 0.0), (129, 131, 77, 0.0), (70, 1, 64, 0.0), (200, 257, 0, 0.0)]


@pytest.mark.parametrize("tb", ["N", "T"])
@pytest.mark.parametrize("variant", [-1, 8, 9, 10])
@pytest.mark.parametrize("mode", [ug.MODE_BF16X1, ug.MODE_BF16X3, ug.MODE_BF16X6, ug.MODE_FP16X3])
def test_problems_without_k_read_no_operand(mode, variant, tb):
    # Ordinary problems of 208 tiles of 128 x 128, four rows of them each: the default splits B in the core.
    full = [Case("R", ta, tb, 500, 3290, 65, 1.5, 0.5, seed=91 + i, pad=i) for i, ta in enumerate("NT")]
    empty = [Case("R", ("N", "T")[i % 2], tb, M, N, K, alpha, (0.25, 0.5, 0.0)[i % 3], seed=97 + i, pad=i % 2)
             for i, (M, N, K, alpha) in enumerate(EMPTY)]
    problems, keep = [], []
    for c in full + empty:
        dC = hip.DeviceArray.from_host(c.C0)
        a = b = None
        if c in full:
            a, b = hip.DeviceArray.from_host(c.A), hip.DeviceArray.from_host(c.B)
        keep.append((c, dC, a, b))
        problems.append(ug.Problem(c.ta.encode(), c.tb.encode(), c.M, c.N, c.K, c.alpha, c.beta, a.ptr if a else None,
                                   c.lda, b.ptr if b else None, c.ldb, dC.ptr, c.ldc))
    ug.force_variant(mode, variant)
    try:
        plan = ug.GroupedPlan(problems, mode=mode, capture=False)
    finally:
        ug.force_variant(mode, -1)
    plan.run(None)
    hip.synchronize()
    for c, dC, a, _ in keep:
        C = dC.download()
        if a:
            ok, worst = c.judge(C, mode=mode)
            assert ok, f"{c.M}x{c.N}x{c.K} {c.ta}{c.tb}: {worst:.3g}"
        else:
            want = c.C0.copy()
            want[:, :c.N] *= np.float32(c.beta)
            assert np.array_equal(C, want), f"{c.M}x{c.N}x{c.K} {c.ta}{c.tb} beta {c.beta}"
    plan.destroy()
