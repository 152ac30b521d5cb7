# SPDX-License-Identifier: Unlicense
"""GPU: 5 x 5 convolutions on the bf16 matrix instructions (at least 16
channels in, 32 out and 96 blocks of 64 channels x 256 pixels, 256 with one
chunk of input channels and more than 32 outputs) against torch's float64
convolution, at the edges of their blocks. Each case asserts that it runs
there (icoreg_conv5_choice).

Bound: as for the products of tests/test_gemm_split_gpu.py, 2^-24 (n / 8 +
16) sum |w x| over the n = 25 C terms, plus the input normalisation's
rounding (three float32 steps a value, 3 * 2^-24 |w x|); for the rms error
2^-24 sqrt((n / 8 + 16) / 3) of the output's rms, the normalisation's three
steps and the bias's two."""

import time

import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

U = 2.0 ** -24
# (images, C, K, H, W, pad, norm, act); act 0 none, 2 ReLU.
CASES = [
    (1, 16, 32, 160, 160, 2, 1, 0),     # one slice of channels, half a block of outputs
    (1, 17, 64, 240, 276, 2, 0, 2),     # a slice with one channel, ragged tiles
    (1, 33, 65, 130, 190, 2, 1, 0),     # 64 channels and one on the few-channel kernel
    (2, 20, 150, 60, 127, 2, 1, 2),     # second block of 128 partly empty, pairs
    (1, 48, 128, 97, 130, 0, 0, 0),     # no padding, pieces over the channels
    (1, 100, 72, 113, 129, 4, 1, 0),    # padding past the window's half, pieces, K = 64 + 8
    (2, 40, 200, 67, 65, 1, 1, 2),
]
# Sizes below those limits: the fp32 instructions.
SMALL = [
    (1, 17, 64, 161, 175, 2, 0, 2),
    (1, 33, 65, 97, 190, 2, 1, 0),
]


def choice(dev, c):
    return dev.api.icoreg_conv5_choice(dev.po, c[0], c[1], c[3], c[4], c[2], c[5])


def tensors(c, seed):
    n, C, K, H, W, pad, norm, act = c
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, C, H, W)).astype(np.float32)
    w = (rng.standard_normal((K, C, 5, 5)) * (2 / (25 * C)) ** 0.5).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, K).astype(np.float32)
    v = [rng.uniform(lo, hi, C).astype(np.float32) for lo, hi in ((-0.2, 0.2), (0.8, 1.25), (0.1, 0.3))]
    return x, w, b, (v if norm else None)


def run(dev, ic, c, x, w, b, v):
    n, C, K, H, W, pad, norm, act = c
    ho, wo = H + 2 * pad - 4, W + 2 * pad - 4
    X, Wt, B = dev.upload(x), dev.upload(w), dev.upload(b)
    V = [dev.upload(t) for t in v] if v else [None] * 3
    out = dev.zeros(n * K * ho * wo)
    g = ic.geom(5, 5, 1, 1, pad, pad, 1, 1, 1)
    dev.api.ops_conv2d_batch(dev.po, n, X.mem, C * H * W, C, H, W, Wt.mem, B.mem, K, ic.C.byref(g),
                             *(ic.mem(t) for t in V), act, 0.0, out.mem, K * ho * wo)
    return dev.read(out).reshape(n, K, ho, wo)


def want(c, x, w, b, v):
    n, C, K, H, W, pad, norm, act = c
    t = torch.from_numpy(x).double()
    if v:
        m, r, a = (torch.from_numpy(q).double()[:, None, None] for q in v)
        t = (t - m) * r
        t = torch.where(t >= 0, t, a * t)
    wd = torch.from_numpy(w).double()
    y = F.conv2d(t, wd, torch.from_numpy(b).double(), padding=pad)
    size = F.conv2d(t.abs(), wd.abs(), torch.from_numpy(b).double().abs(), padding=pad)
    return (y.relu() if act else y).numpy(), size.numpy()


@pytest.mark.parametrize("c", CASES + SMALL, ids=str)
def test_edges(c, dev, ic):
    print(f"[conv split] {c} choice {choice(dev, c)}", flush=True)
    assert (choice(dev, c) > 0) == (c in CASES)
    x, w, b, v = tensors(c, sum(c))
    got = run(dev, ic, c, x, w, b, v)
    ref, size = want(c, x, w, b, v)
    worst = np.max(np.abs(got - ref) / (U * (25 * c[1] / 8 + 19) * size))
    rms = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"[conv split] worst {worst:.3f} of the bound, rms {rms:.2e}", flush=True)
    assert worst <= 1
    if c in CASES:
        assert rms <= U * (((25 * c[1] / 8 + 16) / 3) ** 0.5 + 5)


def test_values_that_are_not_finite(dev, ic):
    c = (1, 18, 40, 240, 276, 2, 0, 0)
    assert choice(dev, c) == 1
    x, w, b, _ = tensors(c, 5)
    x[0, 3, 0, 0] = np.inf
    x[0, 17, 80, 70] = np.nan
    x[0, 0, 239, 275] = 3.4e38  # above the largest bf16
    w[7, 3, 2, 2] = 0           # inf * 0
    w[:, 0] *= 0.5              # no output overflows
    got = run(dev, ic, c, x, w, b, None)
    ref, _ = want(c, x, w, b, None)
    with np.errstate(over="ignore"):
        ref = ref.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    fine = np.isfinite(ref)
    size = np.maximum(np.abs(ref[fine]), 4)
    assert np.max(np.abs(got[fine] - ref[fine]) / size) <= 1e-5


@pytest.mark.parametrize("ex,ew", [(-112, 60), (60, -116), (-120, 0), (-126, 120), (110, -145),
                                   (38, 38), (60, 60)])
def test_magnitudes(ex, ew, dev, ic):
    """Inputs and filters of every size, subnormal ones included, keep their
    24 bits: the sums' rms error is that of the float32 additions, U of a
    partial sum (rms at most the sum's) for each of n / 8 + 16, of random
    sign: U sqrt((n / 8 + 16) / 3). A part lost to bf16's range shows as 2^-22
    of the sum or more."""
    c = (1, 32, 40, 128, 200, 2, 0, 0)
    print(f"[conv split] magnitudes 2^{ex} 2^{ew}", flush=True)
    assert choice(dev, c) == 2
    x, w, b, _ = tensors(c, 3)
    x = np.ldexp(x.astype(np.float64), ex).astype(np.float32)
    w = np.ldexp(w.astype(np.float64), ew).astype(np.float32)
    b[:] = 0
    got = run(dev, ic, c, x, w, b, None)
    ref, _ = want(c, x, w, b, None)
    rms = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    print(f"[conv split] rms error {rms:.2e}", flush=True)
    assert rms <= U * ((25 * c[1] / 8 + 16) / 3) ** 0.5


# Three slices of channels in two pieces; normalised, 128 outputs a block, 16
# and 32 pixels wide tiles.
@pytest.mark.parametrize("c", [(1, 36, 40, 160, 165, 2, 0, 0), (1, 33, 128, 200, 330, 2, 1, 0),
                               (1, 34, 200, 120, 384, 1, 1, 0)], ids=str)
def test_values_that_are_not_finite_again(c, dev, ic):
    """Infinities, NaN and values without a split among the inputs and the
    filters, in the first and the last channels and at corners, come out as
    float32 products give them; outputs they do not reach are unmoved."""
    print(f"[conv split] not finite {c}", flush=True)
    assert choice(dev, c) == (2 if c[1] == 36 else 1)
    x, w, b, v = tensors(c, 11)
    n, C, K, H, W, pad, norm, act = c
    x[0, 3, 0, 0] = np.inf
    x[0, C - 1, H // 2, 70] = np.nan
    x[0, 16, H - 1, W - 1] = 2e38  # above 2^104
    x[0, 5, 30, 100] = -np.inf
    w[7, 3, 2, 2] = 0              # inf * 0
    w[K - 1, 2, 1, 4] = np.inf     # one output channel
    w[:, 16] *= 0.25               # no output overflows
    got = run(dev, ic, c, x, w, b, v)
    with np.errstate(over="ignore", invalid="ignore"):
        ref, size = want(c, x, w, b, v)
        ref = ref.astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    fine = np.isfinite(ref)
    assert fine[0, :K - 1].mean() > 0.9
    # The fp32 instructions round each of the n terms.
    assert np.max(np.abs(got[fine] - ref[fine]) / (U * (25 * C + 19) * size[fine])) <= 1


def test_cost_of_values_that_are_not_finite(dev, ic):
    """A second pass on the fp32 instructions, whose kernel takes about twice
    the bf16 one's time: an image of nothing but NaN costs at most five times
    (a pass that gathers each value took 11)."""
    C, K, H, W = 64, 128, 256, 256
    w = np.ones((K, C, 5, 5), np.float32)
    Wt, B, out = dev.upload(w), dev.zeros(K), dev.zeros(K * H * W)
    g = ic.geom(5, 5, 1, 1, 2, 2, 1, 1, 1)

    def best(value):
        X = dev.upload(np.full((C, H, W), value, np.float32))
        times = []
        for _ in range(6):
            dev.finish()
            t = time.perf_counter()
            for _ in range(5):
                dev.api.ops_conv2d_batch(dev.po, 1, X.mem, C * H * W, C, H, W, Wt.mem, B.mem, K,
                                         ic.C.byref(g), None, None, None, 0, 0.0, out.mem,
                                         K * H * W)
            dev.finish()
            times.append(time.perf_counter() - t)
        return min(times)

    print("[conv split] cost", flush=True)
    assert dev.api.icoreg_conv5_choice(dev.po, 1, C, H, W, K, 2) == 1
    clean, nan = best(1.0), best(np.nan)
    print(f"[conv split] {nan / clean:.2f} times", flush=True)
    assert np.isnan(dev.read(out)).all()
    assert nan <= 5 * clean
