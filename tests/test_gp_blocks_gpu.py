# SPDX-License-Identifier: Unlicense
"""GPU: roma_gp_solve at the edges of its 16-column steps, 16 x 16 tiles and
64-column panels, and the column it reports for a matrix that is not positive
definite.

Bound: the float store rounds by 2^-24. The factorisation works in float64
with reciprocal roots good to 2^-45; its backward error, at most n 2^-45 of
the matrix, is amplified by the condition number (the largest row sum over
the noise, 0.1)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def solve(dev, K, F):
    n, d = F.shape
    bK, bF = dev.upload(K), dev.upload(F)
    work = dev.alloc(int(dev.api.roma_gp_work_bytes(n, d)))
    info = dev.upload(np.full(1, 7, np.int32))
    dev.api.roma_gp_solve(dev.po, bK.mem, n, 0.1, bF.mem, d, work.mem, info.mem)
    return dev.read(bF).reshape(n, d), int(dev.read(info, 1, np.int32)[0])


def kernel(rng, n):
    x = rng.standard_normal((n, 64))
    x /= np.linalg.norm(x, axis=1, keepdims=True)
    return np.exp((x @ x.T - 1) / 0.2).astype(np.float32)


@pytest.mark.parametrize("n", [2, 15, 16, 17, 47, 48, 49, 63, 66, 79, 80, 81, 128, 143, 145, 193])
def test_sizes(n, dev, ic):
    print(f"[gp blocks] n={n}", flush=True)
    rng = np.random.default_rng(n)
    K = kernel(rng, n)
    F = rng.standard_normal((n, 33)).astype(np.float32)
    M = K.astype(np.float64) + np.float64(np.float32(0.1)) * np.eye(n)
    got, info = solve(dev, K, F)
    want = np.linalg.solve(M, F.astype(np.float64))
    cond = np.abs(M).sum(1).max() / 0.1
    bound = 2.0 ** -24 * np.abs(want) + n * 2.0 ** -45 * cond * np.linalg.norm(want, axis=0)
    assert info == 0
    assert np.all(np.abs(got - want) <= bound)


@pytest.mark.parametrize("col", [0, 1, 15, 16, 30, 63, 64, 95, 96, 99])
def test_reports_the_first_bad_column(col, dev, ic):
    n = 100
    K = np.eye(n, dtype=np.float32)
    K[col, col] = -1
    if col + 3 < n:
        K[col + 3, col + 3] = -1
    _, info = solve(dev, K, np.ones((n, 3), np.float32))
    assert info == col + 1
