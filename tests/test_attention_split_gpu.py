# SPDX-License-Identifier: Unlicense
"""GPU: attention on the bf16 matrix instructions against float64 softmax
attention, at the edges of its tiles, key ranges and loads.

Bound: a score's six kept bf16 products lose at most U (d / 8 + 16) of
scale sum |q k| (U = 2^-24: d / 8 additions, the groups' alignment, the
products left out) and the query's scaling 2 U more, so a probability is off
by that much relatively, and by 4 U for its exponential; the numerator and
the denominator both carry it. The sum over the keys adds U (Nk / 8 + 16),
the merge of key ranges and the division 32 U at most, of sum p |v|. That
worst case would hide a lost part, so the rms error is bounded too: scores of
rms 1.5 (at most about 8) have sqrt((d / 8 + 16) / 3) roundings of random sign,
none of more than U of 8 / ln 2; a probability's, its value's and the merge's
are a few U more: within (6 + sqrt(d / 8 + 16)) U of the output's rms. (Small
parts lost in one of the two products make 2^-19 or more.)"""

import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24

# (images, Nq, Nk, heads, d, float offset of the operands, mask)
SHAPES = [
    # One of everything; no channel, key or query tile full.
    (1, 1, 1, 1, 1, 0, 0),
    (1, 33, 31, 3, 5, 0, 1),
    # 32 channels a head, and one to either side; 16-byte loads and not.
    (1, 129, 33, 8, 32, 0, 0),
    (2, 128, 64, 2, 31, 0, 0),
    (1, 127, 65, 2, 33, 0, 1),
    (1, 31, 95, 4, 36, 0, 0),
    (1, 65, 97, 4, 64, 1, 0),
    (2, 400, 400, 8, 32, 0, 0),
    # Key ranges, the last one shorter; few queries over many keys.
    (1, 100, 1000, 8, 64, 0, 1),
    (2, 785, 785, 4, 64, 0, 0),
    # 97 .. 128 channels.
    (1, 40, 130, 2, 97, 0, 0),
    (1, 129, 63, 2, 100, 0, 1),
    (1, 300, 333, 4, 128, 0, 0),
    # No key at all: zeros.
    (1, 40, 0, 2, 64, 0, 0),
]


def run(dev, ic, q, k, v, scale, off=0, mask=None):
    nb, Nq, nh, d = q.shape
    Nk, ld = k.shape[1], nh * d

    def up(x):
        return dev.upload(np.concatenate([np.zeros(off, np.float32), x.ravel(),
                                          np.zeros(4, np.float32)]))

    Q, K, V = up(q), up(k), up(v)
    O = dev.upload(np.full(nb * Nq * ld, 7.0, np.float32))
    keep = dev.upload(mask) if mask is not None else None
    dev.api.ops_attention_batch(dev.po, nb, ic.mat(Q, off, ld), Nq * ld, ic.mat(K, off, ld),
                                Nk * ld, ic.mat(V, off, ld), Nk * ld, ic.mat(O, 0, ld), Nq * ld,
                                Nq, Nk, nh, d, scale, ic.mem(keep) if keep is not None else None)
    return dev.read(O, nb * Nq * ld).reshape(nb, Nq, nh, d)


@pytest.mark.parametrize("shape", SHAPES, ids=[str(s) for s in SHAPES])
def test_edges(shape, dev, ic):
    nb, Nq, Nk, nh, d, off, masked = shape
    print(f"[attention split] {shape}", flush=True)
    rng = np.random.default_rng(Nq + 3 * Nk + d)
    q = rng.standard_normal((nb, Nq, nh, d)).astype(np.float32)
    k = rng.standard_normal((nb, Nk, nh, d)).astype(np.float32)
    v = rng.standard_normal((nb, Nk, nh, d)).astype(np.float32)
    mask = (rng.random(Nk) < 0.7).astype(np.uint8) if masked else None
    scale = float(np.float32(1.5 / np.sqrt(d)))
    got = run(dev, ic, q, k, v, scale, off, mask)
    if Nk == 0:
        assert not got.any()
        return
    qh, kh, vh = (x.astype(np.float64).transpose(0, 2, 1, 3) for x in (q, k, v))
    s = scale * qh @ kh.swapaxes(2, 3)
    size = scale * np.abs(qh) @ np.abs(kh).swapaxes(2, 3)
    if masked:
        s[..., mask == 0] = -np.inf
        size[..., mask == 0] = 0
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    want = (p @ vh).transpose(0, 2, 1, 3)
    rel = 2 * ((d / 8 + 18) * size.max(-1) + 4) + Nk / 8 + 48
    bound = U * (rel[..., None] * (p @ np.abs(vh))).transpose(0, 2, 1, 3)
    worst = np.max(np.abs(got - want) / bound)
    rms = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"[attention split] worst {worst:.3f} of the bound, rms {rms:.2e}", flush=True)
    assert worst <= 1
    assert rms <= U * (6 + (d / 8 + 16) ** 0.5)


@pytest.mark.parametrize("d", [32, 64, 128])
def test_values_that_are_not_finite(d, dev, ic):
    """Infinities, NaN and values above the largest bf16 give what the fp32
    instructions give (a query whose sum of probabilities is NaN gets zeros,
    as one with no key left does); the other heads keep their values."""
    rng = np.random.default_rng(d)
    nh, Nq, Nk = 4, 70, 90
    q, k, v = (rng.standard_normal((1, n, nh, d)).astype(np.float32) for n in (Nq, Nk, Nk))
    scale = float(1.0 / np.sqrt(d))
    clean = run(dev, ic, q, k, v, scale)
    v[0, 88, 0, 3] = np.inf
    v[0, 5, 0, 7] = 3.4e38
    k[0, 40, 1, 0] = np.nan
    q[0, 9, 2, 1] = np.inf
    got = run(dev, ic, q, k, v, scale)[0]
    qh, kh = q[0, :, 0].astype(np.float64), k[0, :, 0].astype(np.float64)
    p = np.exp(scale * qh @ kh.T)
    p /= p.sum(-1, keepdims=True)
    assert np.all(got[:, 0, 3] == np.inf)
    assert np.allclose(got[:, 0, 7], p[:, 5] * 3.4e38, rtol=1e-4)
    assert np.allclose(np.delete(got[:, 0], [3, 7], 1), np.delete(clean[0, :, 0], [3, 7], 1),
                       rtol=0, atol=1e-4)
    assert not got[:, 1].any() and not got[9, 2].any()
    rows = np.delete(np.arange(Nq), 9)
    assert np.allclose(got[rows, 2], clean[0, rows, 2], rtol=0, atol=1e-4)
    assert np.array_equal(got[:, 3], clean[0, :, 3])


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("eq,ek,ev", [(-116, 116, 0), (90, -90, 0), (0, 0, -116), (0, 0, 60),
                                      (-110, 110, -120)])
def test_powers_of_two(eq, ek, ev, d, dev, ic):
    """Scaling queries against keys, or values, by powers of two changes no
    bit but the exponents (no value or result here is subnormal)."""
    print(f"[attention split] 2^{eq} 2^{ek} 2^{ev} d={d}", flush=True)
    rng = np.random.default_rng(d)
    # Magnitudes in [1, 8), values positive: the scaled operands and the
    # results are normal numbers.
    q, k, v = ((rng.uniform(1, 8, (1, n, 2, d)) * rng.choice([-1, 1], (1, n, 2, d))).astype(np.float32)
               for n in (70, 300, 300))
    v = np.abs(v)
    scale = float(np.float32(0.1 / np.sqrt(d)))
    base = run(dev, ic, q, k, v, scale)
    got = run(dev, ic, np.ldexp(q, eq), np.ldexp(k, ek), np.ldexp(v, ev), scale)
    assert np.array_equal(got, np.ldexp(base, ev))


@pytest.mark.parametrize("masked", [0, 1])
@pytest.mark.parametrize("d", [32, 64, 128])
def test_scores_far_below_zero(d, masked, dev, ic):
    """Every score near -2^120: each query takes its best key's values."""
    print(f"[attention split] far below zero d={d} masked={masked}", flush=True)
    rng = np.random.default_rng(d)
    q, k, v = (rng.uniform(0.5, 2, (1, n, 2, d)).astype(np.float32) for n in (70, 300, 300))
    mask = (rng.random(300) < 0.5).astype(np.uint8) if masked else None
    if masked:
        mask[:64] = 0
    got = run(dev, ic, np.ldexp(q, 60), np.ldexp(-k, 60), v, 0.125, 0, mask)
    s = -np.einsum("qhd,khd->hqk", q[0].astype(np.float64), k[0].astype(np.float64))
    if masked:
        s[:, :, mask == 0] = -np.inf
    best = s.argmax(-1)
    for h in range(2):
        assert np.allclose(got[0, :, h], v[0, best[h], h], rtol=4 * U, atol=0)


@pytest.mark.parametrize("d,Nk", [(32, 4000), (64, 4000), (128, 4000)])
def test_positive_values_are_not_biased(d, Nk, dev, ic):
    """Values of one sign: what the small products lose would shift every
    output the same way. The outputs of a query and head share the rounding
    of their denominator, a few U; over 16384 of them the mean's deviation is
    at most 4 U / 128, and it stays within twice that."""
    print(f"[attention split] bias d={d} Nk={Nk}", flush=True)
    rng = np.random.default_rng(5 + d)
    nq, nh = 2048, 8
    q, k = (rng.standard_normal((1, n, nh, d)).astype(np.float32) for n in (nq, Nk))
    v = np.abs(rng.standard_normal((1, Nk, nh, d))).astype(np.float32)
    scale = float(np.float32(1 / np.sqrt(d)))
    got = run(dev, ic, q, k, v, scale)[0]
    shift = 0.0
    for h in range(nh):
        s = scale * q[0, :, h].astype(np.float64) @ k[0, :, h].astype(np.float64).T
        p = np.exp(s - s.max(-1, keepdims=True))
        want = p @ v[0, :, h].astype(np.float64) / p.sum(-1, keepdims=True)
        shift += np.mean(got[:, h] / want - 1) / nh
    print(f"[attention split] mean shift {shift:.2e}", flush=True)
    assert abs(shift) <= U / 16


@pytest.mark.parametrize("d", [32, 64, 128])
def test_values_that_are_not_finite_masked(d, dev, ic):
    """With a key mask: infinities and NaN in keys that are left out change
    nothing but their block's instructions, except a value's, which meets a
    probability of zero (0 * NaN) as in fp32; in keys that are kept they come
    out as without a mask. A key range that is left out whole stays empty."""
    print(f"[attention split] masked not finite d={d}", flush=True)
    rng = np.random.default_rng(d + 1)
    nh, Nq, Nk = 4, 150, 200
    q, k, v = (rng.standard_normal((1, n, nh, d)).astype(np.float32) for n in (Nq, Nk, Nk))
    mask = (rng.random(Nk) < 0.6).astype(np.uint8)
    mask[:64] = 0
    mask[[150, 160]] = 0, 1
    scale = float(1.0 / np.sqrt(d))
    clean = run(dev, ic, q, k, v, scale, 0, mask)[0]
    k[0, 150, 0, 1] = np.nan   # left out
    k[0, 10, 0, 2] = np.inf    # left out
    v[0, 160, 1, 3] = np.inf   # kept
    v[0, 160, 2, 4] = 1e36     # kept, above 2^104
    got = run(dev, ic, q, k, v, scale, 0, mask)[0]
    assert np.allclose(got[:, 0], clean[:, 0], rtol=0, atol=1e-5)
    assert np.all(got[:, 1, 3] == np.inf)
    assert np.allclose(np.delete(got[:, 1], 3, 1), np.delete(clean[:, 1], 3, 1), rtol=0, atol=1e-5)
    s = scale * q[0, :, 2].astype(np.float64) @ k[0, :, 2].astype(np.float64).T
    s[:, mask == 0] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    assert np.allclose(got[:, 2, 4], p[:, 160] * 1e36, rtol=1e-4)
    assert np.array_equal(got[:, 3], clean[:, 3])


def test_cost_of_values_that_are_not_finite(dev, ic):
    """The fp32 block runs after the bf16 one and takes about 1.7 times as
    long: queries of nothing but NaN cost at most 3.3 times (4 without 16-byte
    loads)."""
    nb, n, nh, d = 2, 1601, 8, 128
    ld = nh * d
    K, V = (dev.upload(np.ones((nb, n, ld), np.float32)) for _ in range(2))
    O = dev.zeros(nb * n * ld)

    def best(value):
        Q = dev.upload(np.full((nb, n, ld), value, np.float32))
        times = []
        for _ in range(6):
            dev.finish()
            t = time.perf_counter()
            for _ in range(10):
                dev.api.ops_attention_batch(dev.po, nb, ic.mat(Q, 0, ld), n * ld, ic.mat(K, 0, ld),
                                            n * ld, ic.mat(V, 0, ld), n * ld, ic.mat(O, 0, ld),
                                            n * ld, n, n, nh, d, 0.1, None)
            dev.finish()
            times.append(time.perf_counter() - t)
        return min(times)

    print("[attention split] cost", flush=True)
    clean, nan = best(1.0), best(np.nan)
    print(f"[attention split] {nan / clean:.2f} times", flush=True)
    assert nan <= 3.3 * clean
