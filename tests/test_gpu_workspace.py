"""Workspace kept between calls: calls that need workspace, of sizes that grow
and shrink, from several threads on the null stream and on streams of their
own (created and destroyed on the way, so that handles come back), give the
bits of the no-allocation entry, whose workspace is never shared with them;
a captured call's graph replays right between eager calls; and the library
gives its blocks back at finish and works again after it."""
import ctypes
import threading
import zlib

import numpy as np
import pytest

import ugemm_amd as ug
from ugemm_amd import hip
from tests.helpers import Case

pytestmark = pytest.mark.gpu

# Split-form planes, FP8 planes and split-K partial products, small and larger.
CALLS = [(ug.MODE_FP16X3, 200, 150, 700), (ug.MODE_BF16X3, 512, 600, 900), (ug.MODE_FP32, 64, 64, 5000),
         (ug.MODE_FP8_BLOCK, 300, 257, 500), (ug.MODE_BF16X6, 130, 70, 90), (ug.MODE_FP16X3, 1024, 768, 640)]


class Call:
    def __init__(self, mode, M, N, K):
        self.mode = mode
        self.case = c = Case("R", "N", "N", M, N, K, 1.5, 0.0, seed=zlib.crc32(f"ws{mode}{M},{N},{K}".encode()))
        self.dA, self.dB = hip.DeviceArray.from_host(c.A), hip.DeviceArray.from_host(c.B)
        out = hip.DeviceArray(c.C0.shape, np.float32)
        ug.sgemm_noalloc_dev(*self.args(), out, c.ldc, mode=mode)
        hip.synchronize()
        self.want = out.download().tobytes()

    def args(self):
        c = self.case
        return ("R", "N", "N", c.M, c.N, c.K, c.alpha, self.dA, c.lda, self.dB, c.ldb, 0.0)

    def run(self, out, stream=None):
        ug.sgemm_dev(*self.args(), out, self.case.ldc, mode=self.mode, stream=stream)


@pytest.fixture(scope="module")
def calls():
    return [Call(*c) for c in CALLS]


def rounds(calls, seed, new_stream, wrong):
    order = np.random.default_rng(seed)
    outs = [hip.DeviceArray(c.case.C0.shape, np.float32) for c in calls]
    try:
        for _ in range(12):
            s = hip.Stream() if new_stream else None
            picked = order.permutation(len(calls))
            for i in picked:
                calls[i].run(outs[i], s)
            s.synchronize() if s else hip.synchronize()
            for i in picked:
                if outs[i].download().tobytes() != calls[i].want:
                    wrong.append((seed, int(i)))
            if s:
                s.destroy()
    except Exception as e:   # reported by the test's own thread
        wrong.append(repr(e))


@pytest.mark.parametrize("threads", [1, 4])
def test_calls_of_several_threads_and_streams(calls, threads):
    wrong = []
    ts = [threading.Thread(target=rounds, args=(calls, t, t % 2 == 1, wrong)) for t in range(threads)]
    ts.append(threading.Thread(target=rounds, args=(calls, 77, True, wrong)))
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong, wrong[:5]


def test_captured_call_between_eager_ones(calls):
    L, s = hip.lib(), hip.Stream()
    c, other = calls[1], calls[5]
    out, eager = hip.DeviceArray(c.case.C0.shape, np.float32), hip.DeviceArray(other.case.C0.shape, np.float32)
    c.run(out, s)   # the stream has a block of its own by now
    s.synchronize()
    g, ex = ctypes.c_void_p(), ctypes.c_void_p()
    hip.check(L.hipStreamBeginCapture(ctypes.c_void_p(s.handle), 2), "begin capture")
    try:
        c.run(out, s)
    finally:
        hip.check(L.hipStreamEndCapture(ctypes.c_void_p(s.handle), ctypes.byref(g)), "end capture")
    hip.check(L.hipGraphInstantiate(ctypes.byref(ex), g, None, None, ctypes.c_size_t(0)), "instantiate")
    for _ in range(3):
        out.upload(np.zeros(c.case.C0.shape, np.float32))
        hip.check(L.hipGraphLaunch(ex, ctypes.c_void_p(s.handle)), "launch")
        other.run(eager)
        other.run(eager, s)
        s.synchronize()
        hip.synchronize()
        assert out.download().tobytes() == c.want
        assert eager.download().tobytes() == other.want
    L.hipGraphExecDestroy(ex)
    L.hipGraphDestroy(g)
    s.destroy()


def test_finish_gives_the_blocks_back_and_calls_go_on(calls):
    wrong = []
    rounds(calls[:3], 5, False, wrong)
    ug.finish()
    rounds(calls[:3], 6, True, wrong)
    assert not wrong, wrong[:5]


def test_more_live_streams_than_kept_blocks(calls):
    """70 streams alive at once, three rounds of calls on all of them before
    any is waited for: streams without a kept block allocate as they go."""
    streams = [hip.Stream() for _ in range(70)]
    picked = [calls[i % len(calls)] for i in range(len(streams))]
    outs = [hip.DeviceArray(c.case.C0.shape, np.float32) for c in picked]
    for _ in range(3):
        for c, out, s in zip(picked, outs, streams):
            c.run(out, s)
    for c, out, s in zip(picked, outs, streams):
        s.synchronize()
        assert out.download().tobytes() == c.want
        s.destroy()


def test_finish_beside_running_calls(calls):
    """finish() while calls still run on the caller's stream: their blocks are
    given back only behind them, so other streams' calls change nothing."""
    s, others = hip.Stream(), [hip.Stream() for _ in range(4)]
    outs = [hip.DeviceArray(c.case.C0.shape, np.float32) for c in calls]
    more = [hip.DeviceArray(calls[5].case.C0.shape, np.float32) for _ in others]
    for c, out in zip(calls, outs):
        c.run(out, s)
    ug.finish()
    for o, out in zip(others, more):
        calls[5].run(out, o)
    hip.synchronize()
    assert [out.download().tobytes() == c.want for c, out in zip(calls, outs)] == [True] * len(calls)
    assert all(out.download().tobytes() == calls[5].want for out in more)
    for o in others + [s]:
        o.destroy()
