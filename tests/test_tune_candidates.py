"""What the tuner times, on the CPU: the built-in choice of every product is among
its candidates, also where it takes a split count of its own, so that tuning
makes no product slower."""
import ctypes

import pytest

import ugemm_amd as ug

MODES = [ug.MODE_FP32, ug.MODE_FP32_MFMA, ug.MODE_BF16X1, ug.MODE_BF16X3, ug.MODE_BF16X6, ug.MODE_FP16X3]
SHAPES = [(493, 2304, 34854), (1024, 1024, 4096), (64, 6272, 6592), (5120, 111, 6405), (128, 96, 200),
          (2048, 2048, 2048), (4200, 4200, 2048), (8192, 8192, 512), (1, 1, 100000)]


class Gemm(ctypes.Structure):   # struct Gemm<float> of csrc/internal.h, as far as the choice reads it
    _fields_ = [("M", ctypes.c_int), ("N", ctypes.c_int), ("K", ctypes.c_int), ("alpha", ctypes.c_float),
                ("beta", ctypes.c_float), ("A", ctypes.c_void_p), ("lda", ctypes.c_long), ("B", ctypes.c_void_p),
                ("ldb", ctypes.c_long), ("C", ctypes.c_void_p), ("ldc", ctypes.c_long), ("ta", ctypes.c_bool),
                ("tb", ctypes.c_bool), ("rest", ctypes.c_byte * 256)]


def test_the_built_in_choice_is_timed():
    L, i = ug.load(), ctypes.c_int
    auto = L._ZN5ugemm17automatic_variantERKNS_4GemmIfEEiPi
    candidates = L._ZN5ugemm15tune_candidatesEiiiiiiiPiS0_
    counts = set()
    for mode in MODES:
        for M, N, K in SHAPES:
            for ta in (0, 1):
                for tb in (0, 1):
                    g = Gemm(M, N, K, 1.0, 0.0, None, M if ta else K, None, K if tb else N, None, N, ta, tb)
                    s, vs, ss = i(0), (i * 100)(), (i * 100)()
                    v = auto(ctypes.byref(g), mode, ctypes.byref(s))
                    n = candidates(mode, ta, tb, M, N, K, 100, vs, ss)
                    times = list(zip(vs[:n], ss[:n]))
                    assert times[0] == (v, s.value) and len(set(times)) == n
                    assert {x for x, _ in times} == set(range(len(ug.variants(mode))))
                    counts.add(s.value)
    assert counts - {0, 1, 2, 4, 8, 16}   # counts that the set alone would miss
