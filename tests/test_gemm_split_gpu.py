# SPDX-License-Identifier: Unlicense
"""GPU: ops_gemm and the gathering convolution on the bf16 matrix
instructions (products of more than 512 terms, but for small grids) against
float64 sums, at the edges of their tiles and cuts. Each case states which
instructions it is for (icoreg_gemm_choice).

Bound: a value's six kept bf16 products leave out less than 2^-25 of |a b|;
the matrix core adds groups of eight k, so K / 8 additions round by 2^-24 of
a partial sum that sum |a b| bounds, and a group's alignment drops at most
8 * 2^-24 of its largest product: 2^-24 (K / 8 + 16) sum |a b| in all, and
the float32 epilogue's own 2^-24 a step. That worst case would hide a lost
part, so the rms error is bounded too: of random sign, K / 8 + 16 roundings
of partial sums whose rms is at most the sum's make 2^-24 sqrt((K / 8 + 16) /
3) of it, and the epilogue two more. (The products hl and lh left out make
2^-19 or more.)"""

import time

import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

U = 2.0 ** -24

# (M, N, K, transb, nb, act, residual, biasrow); act 0 none, 2 ReLU, 3 leaky.
SHAPES = [
    # One output, one row, one column; K % 32 != 0.
    (1, 1, 1028, 1, 1, 0, 0, 0),
    (1, 72, 1032, 0, 1, 0, 1, 1),
    (70, 1, 1056, 1, 1, 3, 0, 0),
    # Around one and two 64-row tiles.
    (64, 64, 1056, 1, 1, 0, 0, 0),
    (65, 63, 1028, 1, 1, 2, 0, 1),
    (63, 64, 1060, 0, 1, 0, 1, 0),
    (128, 128, 1056, 0, 2, 0, 1, 0),
    (129, 128, 1060, 0, 1, 3, 0, 1),
    (129, 127, 1060, 1, 1, 3, 0, 1),
    (127, 260, 1140, 0, 3, 2, 1, 0),
    # K just past the rule, 49 tiles of 64 x 64.
    (448, 448, 516, 1, 1, 0, 1, 0),
    (448, 448, 516, 0, 1, 3, 0, 1),
    # Every tile cut over K (few tiles, long K); the last piece shorter.
    (100, 90, 4100, 1, 1, 0, 1, 0),
    (96, 200, 2052, 0, 1, 3, 0, 1),
    # No 16-byte loads: 99 and 121 tiles of 64 x 64 (fewer run elsewhere).
    (700, 520, 577, 1, 1, 2, 1, 0),
    (650, 701, 1023, 0, 1, 0, 0, 1),
    # 64 x 128 tiles.
    (150, 5348, 532, 1, 4, 3, 1, 0),
    (152, 5056, 576, 0, 4, 0, 0, 1),
    # 288 tiles of 128 x 128: 256 whole, 32 cut.
    (2304, 2000, 1024, 1, 1, 0, 1, 0),
]
# Sums of more than 512 terms outside the rule: few tiles, no 16-byte loads or
# under 1024 terms (fp32 instructions).
SMALL = [
    (1, 1, 513, 1, 1, 0, 0, 0),
    (1, 70, 516, 0, 1, 0, 1, 1),
    (70, 1, 544, 1, 1, 3, 0, 0),
    (64, 64, 544, 1, 1, 0, 0, 0),
    (65, 63, 1023, 1, 1, 2, 0, 1),
    (128, 128, 576, 0, 2, 0, 1, 0),
    (129, 127, 577, 0, 1, 3, 0, 1),
]


def run(dev, ic, a, b, shape, alpha, bias, r):
    M, N, K, transb, nb, act, residual, biasrow = shape
    ldb = K if transb else N
    A, B, Bi = dev.upload(a), dev.upload(b), dev.upload(bias)
    out = dev.upload(r)
    dev.api.ops_gemm(dev.po, M, N, K, ic.bmat(A, 0, K, M * K, 0), ic.bmat(B, 0, ldb, N * K, 0),
                     transb, ic.bmat(out, 0, N, M * N, 0), nb, 1, ic.mem(Bi), biasrow,
                     ic.mem(out) if residual else None, 0, alpha, act, 0.1)
    return dev.read(out, nb * M * N).reshape(nb, M, N)


@pytest.mark.parametrize("shape", SHAPES + SMALL, ids=str)
def test_edges(shape, dev, ic):
    M, N, K, transb, nb, act, residual, biasrow = shape
    choice = dev.api.icoreg_gemm_choice(dev.po, M, N, K, transb, nb, 1)
    print(f"[gemm split] {shape} choice {choice}", flush=True)
    assert (choice > 0) == (shape in SHAPES)
    rng = np.random.default_rng(M + 3 * N + K)
    a = rng.standard_normal((nb, M, K)).astype(np.float32)
    b = rng.standard_normal((nb, N, K) if transb else (nb, K, N)).astype(np.float32)
    bias = rng.uniform(-1, 1, M if biasrow else N).astype(np.float32)
    r = rng.uniform(-1, 1, (nb, M, N)).astype(np.float32)
    got = run(dev, ic, a, b, shape, 0.5, bias, r)
    bt = np.swapaxes(b, 1, 2) if transb else b
    v = 0.5 * (a.astype(np.float64) @ bt.astype(np.float64))
    v += bias[:, None] if biasrow else bias
    if act:
        v = np.where(v >= 0, v, (0.0 if act == 2 else 0.1) * v)
    if residual:
        v += r
    size = 0.5 * (np.abs(a).astype(np.float64) @ np.abs(bt).astype(np.float64)) + 2
    worst = np.max(np.abs(got - v) / (U * ((K / 8 + 16) * size + 4 * np.abs(v))))
    rms = np.linalg.norm(got - v) / np.linalg.norm(v)
    print(f"[gemm split] worst {worst:.3f} of the bound, rms {rms:.2e}", flush=True)
    assert worst <= 1
    if choice and M * N >= 64:
        assert rms <= U * (((K / 8 + 16) / 3) ** 0.5 + 2)


@pytest.mark.parametrize("transb", [0, 1])
def test_rows_that_are_not_finite(transb, dev, ic):
    """Infinities, NaN and values that round to bf16 infinity come out as
    float32 products give them, and leave the other rows alone."""
    M, N, K = 200, 152, 1100
    rng = np.random.default_rng(11)
    a = rng.standard_normal((1, M, K)).astype(np.float32)
    b = rng.standard_normal((1, N, K) if transb else (1, K, N)).astype(np.float32)
    a[0, 5, 17] = np.inf
    a[0, 77, 599] = -np.inf
    a[0, 130, 0] = np.nan
    a[0, 190] = 0
    a[0, 190, 3] = 3.4e38  # above the largest bf16
    bt = np.swapaxes(b, 1, 2) if transb else b
    bt[0, 17, 9] = 0  # inf * 0
    with np.errstate(invalid="ignore"):
        v = (a.astype(np.float64) @ bt.astype(np.float64))[0]
    with np.errstate(over="ignore"):
        want = v.astype(np.float32)
    got = run(dev, ic, a, b, (M, N, K, transb, 1, 0, 0, 0), 1.0, np.zeros(N, np.float32),
              np.zeros((1, M, N), np.float32))[0]
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fine = np.isfinite(want)
    rows = np.delete(np.arange(M), [5, 77, 130])
    assert fine[190].any() and np.all(fine[np.delete(rows, rows.searchsorted(190))])
    size = np.abs(a[0, rows]).astype(np.float64) @ np.abs(bt[0]).astype(np.float64)
    off = np.where(fine[rows], np.abs(got[rows] - v[rows]), 0)
    assert np.all(off <= U * (K / 2 + 16) * size)


def test_sums_of_squares_are_not_biased(dev, ic):
    """The Gram diagonal: every term positive, so what the small products
    lose would show as a shift of the mean (it must stay below half a unit
    in the last place)."""
    n, K = 256, 1024
    x = np.random.default_rng(3).standard_normal((1, n, K)).astype(np.float32)
    g = run(dev, ic, x, x, (n, n, K, 1, 1, 0, 0, 0), 1.0, np.zeros(n, np.float32),
            np.zeros((1, n, n), np.float32))[0]
    want = np.sum(x[0].astype(np.float64) ** 2, 1)
    shift = np.mean(np.diag(g) / want - 1)
    print(f"[gemm split] mean shift {shift:.2e}", flush=True)
    assert abs(shift) <= U / 2


@pytest.mark.parametrize("transb", [0, 1])
@pytest.mark.parametrize("ea,eb", [(-112, 60), (60, -116), (-120, 0), (-126, 120), (120, -145),
                                   (-20, -100), (38, 38), (60, 60)])
def test_magnitudes(ea, eb, transb, dev, ic):
    """Operands of every size, subnormal ones included, keep their 24 bits:
    of values of about 2^ea and 2^eb the sums' rms error is that of the
    float32 additions, U of a partial sum (rms at most the sum's) for each of
    K / 8 + 16, of random sign: U sqrt((K / 8 + 16) / 3). A part lost to
    bf16's range shows as 2^-22 of the sum or more."""
    M, N, K = 200, 136, 1100
    print(f"[gemm split] magnitudes 2^{ea} 2^{eb}", flush=True)
    rng = np.random.default_rng(K + ea + 7 * eb)
    a = np.ldexp(rng.standard_normal((1, M, K)), ea).astype(np.float32)
    b = np.ldexp(rng.standard_normal((1, N, K) if transb else (1, K, N)), eb).astype(np.float32)
    got = run(dev, ic, a, b, (M, N, K, transb, 1, 0, 0, 0), 1.0, np.zeros(N, np.float32),
              np.zeros((1, M, N), np.float32))[0]
    bt = (np.swapaxes(b, 1, 2) if transb else b).astype(np.float64)
    want = (a.astype(np.float64) @ bt)[0]
    rms = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"[gemm split] rms error {rms:.2e}", flush=True)
    assert rms <= U * ((K / 8 + 16) / 3) ** 0.5


@pytest.mark.parametrize("transb", [0, 1])
def test_cost_of_values_that_are_not_finite(transb, dev, ic):
    """A second pass on the fp32 instructions, which take about 1.5 times the
    bf16 ones' time: a product of nothing but NaN costs at most four times
    (a pass that gathers each value took 9)."""
    M, N, K = 2048, 2048, 1024
    print(f"[gemm split] cost transb={transb}", flush=True)
    ldb = K if transb else N
    out = dev.zeros(M * N)

    def best(value):
        A = dev.upload(np.full((M, K), value, np.float32))
        B = dev.upload(np.ones((N, K), np.float32))
        times = []
        for _ in range(6):
            dev.finish()
            t = time.perf_counter()
            for _ in range(10):
                dev.api.ops_gemm(dev.po, M, N, K, ic.mat(A, 0, K), ic.mat(B, 0, ldb), transb,
                                 ic.mat(out, 0, N), 1, 1, None, 0, None, 0, 1.0, 0, 0.0)
            dev.finish()
            times.append(time.perf_counter() - t)
        return min(times)

    clean, nan = best(1.0), best(np.nan)
    print(f"[gemm split] {nan / clean:.2f} times", flush=True)
    assert np.isnan(dev.read(out, M * N)).all()
    assert nan <= 4 * clean


# (images, C, K, H, W, window, pad, dilation, stride, norm): more than 512
# terms in shapes that neither the direct nor the Winograd kernels take.
CONVS = [
    (1, 11, 24, 30, 33, 7, 3, 1, 1, 0),    # 539 terms: no 16-byte loads of the filters
    (1, 12, 40, 37, 29, 7, 2, 1, 1, 1),    # 588
    (2, 64, 65, 20, 21, 3, 2, 2, 1, 1),    # dilated, pairs, 576
    (1, 72, 130, 40, 40, 3, 1, 2, 2, 0),
    (1, 3, 70, 112, 84, 14, 0, 1, 14, 0),  # patches, 588
    (1, 130, 200, 64, 70, 3, 2, 2, 1, 1),
]


def conv(dev, ic, c, x, w, b, v):
    n, C, K, H, W, k, pad, dil, stride, norm = c
    ho, wo = ((s + 2 * pad - dil * (k - 1) - 1) // stride + 1 for s in (H, W))
    X, Wt, B, out = dev.upload(x), dev.upload(w), dev.upload(b), dev.zeros(n * K * ho * wo)
    V = [dev.upload(t) for t in v] if norm else [None] * 3
    g = ic.geom(k, k, stride, stride, pad, pad, dil, dil, 1)
    dev.api.ops_conv2d_batch(dev.po, n, X.mem, C * H * W, C, H, W, Wt.mem, B.mem, K, ic.C.byref(g),
                             *(ic.mem(t) for t in V), 0, 0.0, out.mem, K * ho * wo)
    return dev.read(out).reshape(n, K, ho, wo)


@pytest.mark.parametrize("finite", [1, 0])
@pytest.mark.parametrize("c", CONVS, ids=str)
def test_gathered_convolution(c, finite, dev, ic):
    """The input normalised and gated while it is gathered, padding 0; with
    an infinity, a NaN and a value without a split the sums they reach come
    out as float32 products give them (each of K terms rounds)."""
    n, C, K, H, W, k, pad, dil, stride, norm = c
    ho, wo = ((s + 2 * pad - dil * (k - 1) - 1) // stride + 1 for s in (H, W))
    terms = C * k * k
    print(f"[gemm split] conv {c} finite {finite}", flush=True)
    assert dev.api.icoreg_gemm_choice(dev.po, K, ho * wo, terms, 2, n, 1) == 1
    rng = np.random.default_rng(sum(c))
    x = rng.standard_normal((n, C, H, W)).astype(np.float32)
    w = (rng.standard_normal((K, C, k, k)) / terms ** 0.5).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, K).astype(np.float32)
    v = [rng.uniform(lo, hi, C).astype(np.float32) for lo, hi in ((-0.2, 0.2), (0.8, 1.25), (0.1, 0.3))]
    if not finite:
        x[0, 2, 1, 1] = np.inf  # odd places: the strided case reads no other
        x[n - 1, C - 1, H // 4 * 2 + 1, W // 4 * 2 + 1] = np.nan
        x[0, 0, 3, W // 2 * 2 - 5] = 2e38  # above 2^104
        w[3, 2] = 0               # inf * 0
        w[:, 0] *= 0.25           # no output overflows
    got = conv(dev, ic, c, x, w, b, v)
    t = torch.from_numpy(x).double()
    if norm:
        m, r, a = (torch.from_numpy(q).double()[:, None, None] for q in v)
        t = (t - m) * r
        t = torch.where(t >= 0, t, a * t)
    args = {"padding": pad, "dilation": dil, "stride": stride}
    wd, bd = torch.from_numpy(w).double(), torch.from_numpy(b).double()
    want = F.conv2d(t, wd, bd, **args).numpy()
    size = F.conv2d(t.abs(), wd.abs(), bd.abs(), **args).numpy()
    if finite:
        worst = np.max(np.abs(got - want) / (U * (terms / 8 + 19) * size))
        rms = np.linalg.norm(got - want) / np.linalg.norm(want)
        print(f"[gemm split] worst {worst:.3f} of the bound, rms {rms:.2e}", flush=True)
        assert worst <= 1 and rms <= U * (((terms / 8 + 16) / 3) ** 0.5 + 5)
        return
    with np.errstate(over="ignore"):
        want32 = want.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want32))
    assert np.array_equal(got[np.isinf(want32)], want32[np.isinf(want32)])
    fine = np.isfinite(want32)
    assert fine.any() and not fine.all()
    assert np.max(np.abs(got[fine] - want[fine]) / (U * (terms + 19) * size[fine])) <= 1
