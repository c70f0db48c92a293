"""The work that callers of this library have it do, as measurable cases.

Every case goes through a public entry point of ugemm_amd with operands that
already lie on the GPU: a matrix product in one of the arithmetic forms, an
FP64 product, a planned batch of uneven products, a batch of convolutions (or
one), a matrix-vector product.  listed() names the ones that are followed;
draw() gives others of the same kinds and ranges: every form and layout, both
majors, padded leading dimensions, ragged sizes, tall, wide and deep shapes.
"""
import math
import random

import numpy as np
import torch
import torch.nn.functional as F

import ugemm_amd as ug

# A drawn product has at most this many floating-point operations (2 M N K),
# and an operand at most this many elements.
MAX_FLOP = {"gemm": 2.7e11, "dgemm": 1.3e11}
MAX_ELEMENTS = 1 << 28
# The forms, with how often a drawn product uses each: the FP32-accuracy ones
# mostly, the low-precision ones now and then.
FORMS = (("fp32", 30), ("fp16x3", 30), ("bf16x3", 16), ("fp32_mfma", 10), ("bf16x6", 6), ("bf16x1", 4), ("fp8", 4))


def _gemm(name, mode, ta, tb, M, N, K, alpha, beta, dist="uniform"):
    return {"name": name, "kind": "gemm", "mode": mode, "major": "R", "ta": ta, "tb": tb, "M": M, "N": N, "K": K,
            "alpha": alpha, "beta": beta, "pad": 0, "dist": dist}


def listed():
    return [
        # A call whose cost is latency and launches: a small product inside a caller's loop.
        _gemm("sgemm_small", "fp32", "N", "N", 128, 96, 200, 1.0, 0.0),
        # The size of the reference's own GPU test program (no dimension of the operands aligned).
        _gemm("sgemm_1023x1000x1023", "fp32", "N", "N", 1023, 1000, 1023, 1.0, 0.0),
        # An ordinary large product in the plain form, accumulating into C.
        _gemm("sgemm_4096", "fp32", "N", "N", 4096, 4096, 4096, 1.5, 0.5),
        # The headline: FP32-level error on the 16-bit matrix cores at 8192^3.
        _gemm("fp16x3_8192", "fp16x3", "N", "N", 8192, 8192, 8192, 1.5, 0.5),
        # The same form at an ordinary size, B transposed (a layer's weights stored output by input).
        _gemm("fp16x3_2048_nt", "fp16x3", "N", "T", 2048, 2048, 2048, 1.0, 0.0),
        # Tall and skinny: a long list of rows through one narrow layer.
        _gemm("bf16x3_tall", "bf16x3", "N", "N", 65536, 256, 4096, 1.0, 0.0, "normal"),
        # A transposed and K long: the product that gives a layer's weight gradient, added up over calls.
        _gemm("fp32_mfma_deep_tn", "fp32_mfma", "T", "N", 576, 384, 50176, 1.0, 1.0, "normal"),
        # FP64.
        {"name": "dgemm_4096", "kind": "dgemm", "major": "R", "ta": "N", "tb": "N", "M": 4096, "N": 4096, "K": 4096,
         "alpha": 1.0, "beta": 0.0, "pad": 0, "dist": "normal"},
        # Batches of uneven im2col-shaped products, planned once and replayed, in the plain form and
        # in the one with FP32-level error on the matrix cores.
        {"name": "grouped_fp32_512", "kind": "grouped", "mode": "fp32", "count": 512, "tb": "N", "ragged": False,
         "shapes": 4},
        {"name": "grouped_fp16x3_512", "kind": "grouped", "mode": "fp16x3", "count": 512, "tb": "N", "ragged": False,
         "shapes": 4},
        # The convolutions of a network (3x3, pad 1, bias, LeakyReLU), planned once and replayed.
        {"name": "conv_128", "kind": "conv", "mode": "fp32", "count": 128, "k": 3, "pad": 1, "stride": 1,
         "ragged": False, "shapes": 4},
        # A fully connected layer on one input.
        {"name": "sgemv_t_8192", "kind": "gemv", "dtype": "f32", "trans": "T", "M": 8192, "N": 8192, "alpha": 1.0,
         "beta": 0.0, "pad": 0},
    ]


def _size(rng, lo, hi):
    """A size between lo and hi, spread over the logarithm; half of them multiples of 64 where that fits."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 64 and rng.random() < 0.5:
        v = max(64, v // 64 * 64)
    return max(lo, min(hi, v))


def _weighted(rng, table):
    return rng.choices([x for x, _ in table], [w for _, w in table])[0]


def draw(rng):
    kind = _weighted(rng, (("gemm", 52), ("dgemm", 10), ("grouped", 14), ("conv", 12), ("gemv", 12)))
    if kind in ("gemm", "dgemm"):
        dims = [_size(rng, 24, 8192) for _ in range(3)]
        if rng.random() < 0.3:   # one long side: tall, wide or deep
            dims[rng.randrange(3)] = _size(rng, 4096, 65536)
        while (2.0 * dims[0] * dims[1] * dims[2] > MAX_FLOP[kind]
               or max(dims[0] * dims[2], dims[2] * dims[1], dims[0] * dims[1]) > MAX_ELEMENTS):
            i = max(range(3), key=lambda d: dims[d])
            dims[i] = dims[i] * 3 // 4
        alpha, beta = rng.choice(((1.0, 0.0), (1.0, 0.0), (1.5, 0.5), (1.0, 1.0)))
        case = {"kind": kind, "major": rng.choice("RRRRC"), "ta": rng.choice("NNT"), "tb": rng.choice("NNT"),
                "M": dims[0], "N": dims[1], "K": dims[2], "alpha": alpha, "beta": beta,
                "pad": rng.choice((0, 0, 0, 8, 3)), "dist": rng.choice(("uniform", "normal"))}
        if kind == "gemm":
            case["mode"] = _weighted(rng, FORMS)
        return case
    if kind == "grouped":
        return {"kind": kind, "mode": rng.choice(("fp32", "fp32", "fp16x3", "fp16x3", "bf16x3", "fp32_mfma")),
                "count": _size(rng, 4, 400), "tb": rng.choice("NNT"), "ragged": rng.random() < 0.5,
                "shapes": rng.randrange(1 << 16)}
    if kind == "conv":
        k, pad, stride = rng.choice(((3, 1, 1), (3, 1, 1), (1, 0, 1), (3, 1, 2), (5, 2, 2)))
        mode = rng.choice(("fp32", "fp32", "fp32_mfma"))
        return {"kind": kind, "mode": mode, "count": rng.choice((1, 1, _size(rng, 2, 128))), "k": k, "pad": pad,
                "stride": stride, "ragged": rng.random() < 0.5, "shapes": rng.randrange(1 << 16)}
    M, N = _size(rng, 64, 32768), _size(rng, 64, 32768)
    while M * N > MAX_ELEMENTS // 2:
        M = M * 3 // 4
    return {"kind": kind, "dtype": rng.choice(("f32", "f32", "f64")), "trans": rng.choice("NT"), "M": M, "N": N,
            "alpha": rng.choice((1.0, 0.5)), "beta": rng.choice((0.0, 1.0)), "pad": rng.choice((0, 0, 8, 3))}


# ---------------------------------------------------------------------------
# Shapes and inputs.
def _problems(case):
    """(M, N, K) of every product of a batch: M output channels, N output pixels, K = 9 x input channels."""
    g = random.Random(case["shapes"])
    out = []
    for _ in range(case["count"]):
        if case["ragged"]:
            out.append((g.randint(17, 512), g.randint(5, 60) ** 2, 9 * g.randint(3, 512)))
        else:
            out.append((32 * g.randint(1, 16), g.choice((7, 14, 28, 56)) ** 2, 144 * g.randint(1, 32)))
    return out


def _convs(case):
    """(ich, h, w, ch, hcol, wcol) of every convolution of a batch."""
    g = random.Random(case["shapes"])
    out = []
    for _ in range(case["count"]):
        if case["ragged"]:
            ich, h, w, ch = g.randint(3, 300), g.randint(9, 60), g.randint(9, 60), g.randint(10, 400)
        else:
            ich, h, ch = 16 * g.randint(1, 32), g.choice((7, 14, 28, 56)), 32 * g.randint(1, 16)
            w = h
        out.append((ich, h, w, ch, (h + 2 * case["pad"] - case["k"]) // case["stride"] + 1,
                    (w + 2 * case["pad"] - case["k"]) // case["stride"] + 1))
    return out


def _offsets(sizes):
    """Start of every buffer in one allocation (256-byte aligned), and its length."""
    return np.concatenate([[0], np.cumsum([(n + 63) // 64 * 64 for n in sizes])]).astype(np.int64)


def _values(g, shape, dist, dtype=torch.float32):
    if dist == "normal":
        return torch.randn(shape, generator=g, device="cuda", dtype=dtype)
    return torch.rand(shape, generator=g, device="cuda", dtype=dtype).mul_(2.0).sub_(1.0)


def _a_by_k(case):
    """Whether A is stored as K rows of M values (else M rows of K): transposed, or column-major, not both."""
    return (case["ta"] == "T") != (case["major"] == "C")


def _b_by_n(case):
    """Whether B is stored as N rows of K values (else K rows of N)."""
    return (case["tb"] == "T") != (case["major"] == "C")


def _inputs(case, seed):
    """The operands of a case, from the seed alone."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    kind = case["kind"]
    if kind in ("gemm", "dgemm"):
        dtype = torch.float64 if kind == "dgemm" else torch.float32
        M, N, K, pad = case["M"], case["N"], case["K"], case["pad"]
        flip = case["major"] == "C"
        a = (K, M) if _a_by_k(case) else (M, K)   # stored rows and row length
        b = (N, K) if _b_by_n(case) else (K, N)
        c = (N, M) if flip else (M, N)
        A = _values(g, (a[0], a[1] + pad), case["dist"], dtype)
        B = _values(g, (b[0], b[1] + pad), case["dist"], dtype)
        C = torch.zeros((c[0], c[1] + pad), device="cuda", dtype=dtype)
        if case["beta"] != 0.0:
            C = _values(g, C.shape, case["dist"], dtype)
        return {"A": A, "B": B, "C": C}
    if kind == "grouped":
        P = _problems(case)
        ao, bo, co = (_offsets([f(p) for p in P]) for f in (lambda p: p[0] * p[2], lambda p: p[2] * p[1],
                                                             lambda p: p[0] * p[1]))
        return {"A": _values(g, int(ao[-1]), "uniform"), "B": _values(g, int(bo[-1]), "uniform"),
                "C": torch.zeros(int(co[-1]), device="cuda"), "problems": P, "ao": ao, "bo": bo, "co": co}
    if kind == "conv":
        P, k = _convs(case), case["k"]
        xo = _offsets([p[0] * p[1] * p[2] for p in P])
        wo = _offsets([p[3] * p[0] * k * k for p in P])
        bo = _offsets([p[3] for p in P])
        oo = _offsets([p[3] * p[4] * p[5] for p in P])
        x = _values(g, int(xo[-1]), "normal")
        wts = _values(g, int(wo[-1]), "normal")
        for i, p in enumerate(P):   # weights of the size a trained layer's have
            wts[int(wo[i]):int(wo[i + 1])] *= (p[0] * k * k) ** -0.5
        return {"x": x, "w": wts, "b": _values(g, int(bo[-1]), "normal"), "o": torch.zeros(int(oo[-1]), device="cuda"),
                "convs": P, "xo": xo, "wo": wo, "bo": bo, "oo": oo}
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float32
    M, N, pad = case["M"], case["N"], case["pad"]
    A = _values(g, (M, N + pad) if case["trans"] == "T" else (N, M + pad), "normal", dtype)
    x = _values(g, N, "normal", dtype)
    y = torch.zeros(M, device="cuda", dtype=dtype)
    if case["beta"] != 0.0:
        y = _values(g, M, "normal", dtype)
    return {"A": A, "x": x, "y": y}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "grouped":
        # The plan a program makes once for its batch; it keeps the operands' addresses.
        a, b, c = s["A"].data_ptr(), s["B"].data_ptr(), s["C"].data_ptr()
        tb = case["tb"]
        s["plan"] = ug.GroupedPlan(
            [ug.Problem(b"N", tb.encode(), M, N, K, 1.0, 0.0, a + 4 * int(s["ao"][i]), K, b + 4 * int(s["bo"][i]),
                        K if tb == "T" else N, c + 4 * int(s["co"][i]), N)
             for i, (M, N, K) in enumerate(s["problems"])], mode=ug.MODES[case["mode"]], capture=True)
    elif case["kind"] == "conv" and case["count"] > 1:
        x, w, b, o = (s[n].data_ptr() for n in "xwbo")
        s["plan"] = ug.GroupedPlan(
            [ug.ConvProblem(x + 4 * int(s["xo"][i]), ich, wd, h, w + 4 * int(s["wo"][i]), case["k"], case["pad"],
                            case["stride"], o + 4 * int(s["oo"][i]), ch, b + 4 * int(s["bo"][i]),
                            ug.ACT_LEAKY_RELU, 0.1)
             for i, (ich, h, wd, ch, _, _) in enumerate(s["convs"])], mode=ug.MODES[case["mode"]], capture=True)
    return s


def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "gemm":
        A, B, C = s["A"], s["B"], s["C"]
        ug.sgemm_dev(c["major"], c["ta"], c["tb"], c["M"], c["N"], c["K"], c["alpha"], A.data_ptr(), A.shape[1],
                     B.data_ptr(), B.shape[1], c["beta"], C.data_ptr(), C.shape[1], mode=ug.MODES[c["mode"]])
        return C
    if kind == "dgemm":
        A, B, C = s["A"], s["B"], s["C"]
        ug.dgemm_dev(c["major"], c["ta"], c["tb"], c["M"], c["N"], c["K"], c["alpha"], A.data_ptr(), A.shape[1],
                     B.data_ptr(), B.shape[1], c["beta"], C.data_ptr(), C.shape[1])
        return C
    if kind == "grouped":
        s["plan"].run()
        return s["C"]
    if kind == "conv":
        if "plan" in s:
            s["plan"].run()
        else:
            ich, h, w, ch, _, _ = s["convs"][0]
            ug.conv2d_dev(s["x"].data_ptr(), ich, w, h, s["w"].data_ptr(), c["k"], c["pad"], c["stride"],
                          s["o"].data_ptr(), ch, bias=s["b"].data_ptr(), act=ug.ACT_LEAKY_RELU, slope=0.1,
                          mode=ug.MODES[c["mode"]])
        return s["o"]
    ug.gemv_dev(c["trans"], c["M"], c["N"], c["alpha"], s["A"].data_ptr(), s["A"].shape[1], s["x"].data_ptr(), 1,
                c["beta"], s["y"].data_ptr(), 1, double=c["dtype"] == "f64")
    return s["y"]


def work(case):
    kind = case["kind"]
    if kind in ("gemm", "dgemm"):
        M, N, K = case["M"], case["N"], case["K"]
        size = 8 if kind == "dgemm" else 4
        return {"bytes": size * (M * K + K * N + M * N * (2 if case["beta"] != 0.0 else 1)), "flops": 2.0 * M * N * K}
    if kind == "grouped":
        P = _problems(case)
        return {"bytes": 4 * sum(M * K + K * N + M * N for M, N, K in P), "flops": sum(2.0 * M * N * K for M, N, K in P)}
    if kind == "conv":
        P, kk = _convs(case), case["k"] ** 2
        return {"bytes": 4 * sum(p[0] * p[1] * p[2] + p[3] * p[0] * kk + p[3] + p[3] * p[4] * p[5] for p in P),
                "flops": sum(2.0 * p[3] * p[4] * p[5] * p[0] * kk for p in P)}
    M, N = case["M"], case["N"]
    size = 8 if case["dtype"] == "f64" else 4
    return {"bytes": size * (M * N + N + M * (2 if case["beta"] != 0.0 else 1)), "flops": 2.0 * M * N}


def exact(case, seed):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("gemm", "dgemm"):
        M, N, K, flip = case["M"], case["N"], case["K"], case["major"] == "C"
        A, B, C = s["A"].double(), s["B"].double(), s["C"].double()
        # op(A) (M x K) and op(B) (K x N); a column-major matrix is its transpose's rows.
        a = A[:, :M].t() if _a_by_k(case) else A[:, :K]
        b = B[:, :K].t() if _b_by_n(case) else B[:, :N]
        c = C[:, :M].t() if flip else C[:, :N]
        c.copy_(case["alpha"] * (a @ b) + case["beta"] * c)
        return C
    if kind == "grouped":
        out = torch.zeros_like(s["C"], dtype=torch.float64)
        for i, (M, N, K) in enumerate(s["problems"]):
            a = s["A"][int(s["ao"][i]):][:M * K].view(M, K).double()
            b = s["B"][int(s["bo"][i]):][:K * N].double()
            b = b.view(N, K).t() if case["tb"] == "T" else b.view(K, N)
            out[int(s["co"][i]):][:M * N] = (a @ b).reshape(-1)
        return out
    if kind == "conv":
        out = torch.zeros_like(s["o"], dtype=torch.float64)
        k = case["k"]
        for i, (ich, h, w, ch, hc, wc) in enumerate(s["convs"]):
            x = s["x"][int(s["xo"][i]):][:ich * h * w].view(1, ich, h, w).double()
            wt = s["w"][int(s["wo"][i]):][:ch * ich * k * k].view(ch, ich * k * k).double()
            col = F.unfold(x, k, padding=case["pad"], stride=case["stride"])[0]
            v = wt @ col + s["b"][int(s["bo"][i]):][:ch].double()[:, None]
            # The layer's slope is a float32 value.
            out[int(s["oo"][i]):][:ch * hc * wc] = torch.where(v > 0, v, v * float(np.float32(0.1))).reshape(-1)
        return out
    A = s["A"].double()
    A = A[:, :case["N"]] if case["trans"] == "T" else A[:, :case["M"]].t()
    return case["alpha"] * (A @ s["x"].double()) + case["beta"] * s["y"].double()
