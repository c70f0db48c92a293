"""Workspace blocks kept between calls, on the CPU: the library's allocator over
stand-ins for the HIP calls (c_harness/fake_hip_memory.c).  A call never waits
(hipFree) for another stream, whatever the number of streams and sizes; what
is kept stays within its bounds; the null stream keeps its own."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

from ugemm_amd.build import LIB

HERE = os.path.dirname(os.path.abspath(__file__))
MIB = 1 << 20

# In a process of its own: the stand-ins are in front of the runtime there.
PRELUDE = """
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
L = ctypes.CDLL(sys.argv[2])
alloc, free = L._ZN5ugemm12stream_allocEPPvmP12ihipStream_t, L._ZN5ugemm11stream_freeEPvP12ihipStream_t
alloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_void_p]
free.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
MIB = 1 << 20
counter = lambda name: ctypes.c_int.in_dll(fake, "fake_" + name)
size = lambda name: ctypes.c_size_t.in_dll(fake, "fake_" + name)
count = lambda: tuple(counter(n).value for n in ("mallocs", "frees_async", "frees"))
def call(nbytes, stream, status=0):
    p = ctypes.c_void_p()
    rc = alloc(ctypes.byref(p), nbytes, stream)
    assert rc == status, rc
    assert bool(p.value) == (status == 0)
    return p.value
def once(nbytes, stream):
    p = call(nbytes, stream)
    assert free(p, stream) == 0
    return p
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None or not os.path.exists(LIB):
        pytest.skip("no C compiler, or libugemm_hip.so is not built")
    so = str(tmp_path_factory.mktemp("fake") / "libfake_hip_memory.so")
    subprocess.run([cc, "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "c_harness", "fake_hip_memory.c")], check=True)
    return so


def run(fake, body):
    code = PRELUDE + textwrap.dedent(body) + "\nassert counter('wrong').value == 0\nprint('done')\n"
    r = subprocess.run([sys.executable, "-c", code, fake, LIB], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "done", r.stderr


def test_a_stream_gets_its_block_back(fake):
    run(fake, """
        a = once(5 * MIB, 101)
        assert once(3 * MIB, 101) == a and count() == (1, 0, 0)
        b = once(9 * MIB, 101)                      # too small: replaced, in the stream's own order
        assert once(5 * MIB, 101) == b and count() == (2, 1, 0)
        p, q = call(MIB, 101), call(MIB, 101)         # two calls at once
        assert p != q and free(p, 101) == 0 and free(q, 101) == 0
        """)


def test_many_streams_never_wait(fake):
    """80 streams in turn, each time from the first on: those without a place
    allocate and free in stream order, and no block changes its stream."""
    run(fake, """
        for turn in range(3):
            for s in range(100, 180):
                once(2 * MIB, s)
        assert count() == (56 + 3 * 24, 3 * 24, 0) and size("bytes").value == 56 * 2 * MIB
        a = once(100 * MIB, 0)                    # the null stream still keeps its block
        assert once(MIB, 0) == a
        """)


def test_large_blocks_never_wait(fake):
    """Five streams of 120 MiB pass the 512 MiB that may be kept."""
    run(fake, """
        for turn in range(3):
            for s in (101, 102, 103, 104, 105, 0):
                once(120 * MIB, s)
        assert count()[2] == 0 and size("bytes").value == 4 * 120 * MIB
        assert once(MIB, 0) == once(120 * MIB, 0) # the null stream's is among them
        once(200 * MIB, 101)                      # beyond a kept block's size
        assert count()[2] == 0 and size("bytes").value == 4 * 120 * MIB
        """)


def test_idle_blocks_are_released_after_a_wait_and_kept_if_refused(fake):
    run(fake, """
        release = L._ZN5ugemm22release_idle_workspaceEv
        a, b = once(3 * MIB, 101), once(4 * MIB, 0)
        p = call(MIB, 102)                        # in use: stays
        counter("refuse").value = 1
        assert release() == 0 and once(3 * MIB, 101) == a and once(4 * MIB, 0) == b
        c = call(9 * MIB, 101)                    # a is not replaced: the call has memory of its own
        counter("refuse").value = 0
        assert free(c, 101) == 0 and once(2 * MIB, 101) == a
        assert release() == 2 and size("bytes").value == MIB
        assert free(p, 102) == 0 and release() == 1 and size("bytes").value == 0
        """)


@pytest.mark.parametrize("large", [100, 300])
def test_a_call_out_of_memory_takes_back_the_idle_blocks(fake, large):
    """What fits without kept blocks fits beside them: of a size that is kept
    and of one that is not."""
    run(fake, f"""
        size("limit").value = 350 * MIB
        for s in (101, 102, 0):
            once(100 * MIB, s)
        p = call(MIB, 103)                        # in use: stays
        q = call({large} * MIB, 104)
        assert count()[2] == 3 and size("bytes").value == {large + 1} * MIB
        call(400 * MIB, 105, status=-3)           # nothing left to give back
        assert free(q, 104) == 0 and free(p, 103) == 0
        once(100 * MIB, 101)
        """)
