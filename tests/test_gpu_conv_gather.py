"""The im2col gather of the FP32 and FP32-MFMA convolutions and the choices
around it: kernels of 1 to 49 taps (on both sides of the 32 whose bounds are
kept as bits), strides and paddings that put whole rows of taps outside the
image, K around the 16-deep steps and the groups of a workgroup, channel counts
around the tiles; alone and in plans of few, some and many tiles; 1x1
convolutions, which run as plain products.  Against the oracle's convolution
and the FP32 bound."""
import zlib

import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# ich, h, w, k, pad, stride, ch
SHAPES = [
    (1, 1, 1, 1, 0, 1, 1), (5, 9, 7, 1, 0, 1, 33), (64, 15, 13, 1, 0, 1, 65), (7, 11, 10, 1, 0, 2, 12),
    (3, 6, 5, 2, 1, 1, 31), (1, 4, 4, 3, 2, 1, 2), (5, 12, 9, 3, 1, 3, 64), (29, 17, 16, 3, 1, 1, 66),
    (4, 8, 9, 5, 2, 1, 40), (2, 13, 12, 5, 4, 2, 7), (3, 9, 9, 6, 3, 1, 32), (2, 16, 14, 7, 3, 2, 34),
    (130, 7, 7, 3, 1, 1, 130), (300, 5, 6, 3, 1, 1, 20), (2, 90, 80, 3, 1, 1, 10), (16, 60, 61, 3, 1, 1, 200),
]
MODES = [ug.MODE_FP32, ug.MODE_FP32_MFMA]


def operands(shape, seed):
    ich, h, w, k, pad, stride, ch = shape
    g = orc.rng(zlib.crc32(f"gather{shape}{seed}".encode()))
    return orc.uniform(g, (ich, h, w)), orc.uniform(g, (ch, ich * k * k)), orc.uniform(g, (ch,))


def check(got, shape, x, wts, bias):
    ich, h, w, k, pad, stride, ch = shape
    col = orc.im2col(x, ich, h, w, k, pad, stride).astype(np.float64).reshape(ich * k * k, -1)
    pre = wts.astype(np.float64) @ col + bias[:, None]
    want = np.where(pre > 0, pre, np.float64(np.float32(0.1)) * pre)
    scale = np.abs(wts).astype(np.float64) @ np.abs(col) + np.abs(bias)[:, None]
    err = np.abs(got.reshape(ch, -1) - want)
    assert np.all(err <= orc.tolerance(ich * k * k + 2) * scale), f"{shape}: {np.max(err / (scale + 1e-30)):.3g}"


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("shape", SHAPES)
def test_single_convolutions(mode, shape):
    ich, h, w, k, pad, stride, ch = shape
    x, wts, bias = operands(shape, mode)
    hc, wc = orc.conv_out_shape(h, w, k, pad, stride)
    dx, dw, db = (hip.DeviceArray.from_host(a) for a in (x, wts, bias))
    do = hip.DeviceArray.from_host(np.full((ch, hc * wc), np.nan, np.float32))
    for variant in (-1, 0, 1, 2, 3):
        print(f"mode {mode} {shape} variant {variant}", flush=True)
        ug.force_variant(mode, variant)
        try:
            ug.conv2d_dev(dx, ich, w, h, dw, k, pad, stride, do, ch, bias=db, mode=mode)
        finally:
            ug.force_variant(mode, -1)
        hip.synchronize()
        check(do.download(), shape, x, wts, bias)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("copies", [1, 3, 40])
def test_plans_of_convolutions(mode, copies):
    """All shapes in one plan, `copies` times (few tiles: groups of a
    workgroup; many: one group), twice in a row."""
    problems, bufs = [], []
    for c in range(copies):
        for shape in SHAPES:
            ich, h, w, k, pad, stride, ch = shape
            x, wts, bias = operands(shape, c % 3)
            hc, wc = orc.conv_out_shape(h, w, k, pad, stride)
            dx, dw, db = (hip.DeviceArray.from_host(a) for a in (x, wts, bias))
            do = hip.DeviceArray.from_host(np.full((ch, hc * wc), np.nan, np.float32))
            bufs.append((shape, x, wts, bias, dx, dw, db, do))
            problems.append(ug.ConvProblem(dx.ptr, ich, w, h, dw.ptr, k, pad, stride, do.ptr, ch, db.ptr,
                                           ug.ACT_LEAKY_RELU, 0.1))
    plan = ug.GroupedPlan(problems, mode=mode, capture=True)
    for _ in range(2):
        plan.run()
        hip.synchronize()
    for shape, x, wts, bias, dx, dw, db, do in bufs[:len(SHAPES)] + bufs[-len(SHAPES):]:
        check(do.download(), shape, x, wts, bias)
    plan.destroy()


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("count", [1, 6, 30, 200])
@pytest.mark.parametrize("tb", ["N", "T"])
def test_plans_of_few_and_many_products(mode, count, tb):
    """Uneven products around the tiles' edges: groups of 8 and 4, one group,
    and (FP32) a row remainder of up to 64 and of more than 64 below 128-row
    tiles, through every variant."""
    g = orc.rng(7 * count + mode)
    Ms, Ns, Ks = (g.integers(1, hi, size=count) for hi in (420, 500, 300))
    Ks[0] = 1200
    items = []
    for M, N, K in zip(Ms, Ns, Ks):
        A, B = orc.uniform(g, (int(M), int(K))), orc.uniform(g, (int(N), int(K)) if tb == "T" else (int(K), int(N)))
        items.append((A, B, hip.DeviceArray.from_host(A), hip.DeviceArray.from_host(B),
                      hip.DeviceArray((int(M), int(N)), np.float32)))
    for variant in (-1, 1, 4, 0):
        ug.force_variant(mode, variant)
        try:
            plan = ug.GroupedPlan([ug.Problem(b"N", tb.encode(), A.shape[0], dC.shape[1], A.shape[1], 1.0, 0.0, dA.ptr,
                                              A.shape[1], dB.ptr, B.shape[1], dC.ptr, dC.shape[1])
                                   for A, B, dA, dB, dC in items], mode=mode)
        finally:
            ug.force_variant(mode, -1)
        print(f"mode {mode} count {count} {tb} variant {variant}", flush=True)
        plan.run()
        hip.synchronize()
        for A, B, dA, dB, dC in items:
            Bk = (B.T if tb == "T" else B).astype(np.float64)
            err = np.abs(dC.download() - A.astype(np.float64) @ Bk)
            scale = np.abs(A).astype(np.float64) @ np.abs(Bk)
            assert np.all(err <= orc.tolerance(A.shape[1]) * scale), (variant, A.shape, B.shape)
        plan.destroy()
