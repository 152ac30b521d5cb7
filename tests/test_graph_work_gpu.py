# SPDX-License-Identifier: Unlicense
"""GPU: products and 5 x 5 convolutions recorded into a graph before the ops
work buffer has the size of their bf16 kernel. Where the fp32 kernel needs
none of it, the call is recorded with that one; where it needs some too, the
call is refused, and the device works on."""

import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture
def fresh(ic):
    """A device whose work buffer is empty."""
    d = ic.Device("auto")
    yield d
    d.close()


def gemm(d, ic, M, N, K):
    """A run function, its output buffer and the float64 result."""
    rng = np.random.default_rng(M + K)
    a, b = (rng.standard_normal((n, K)).astype(np.float32) for n in (M, N))
    A, B, out = d.upload(a), d.upload(b), d.zeros(M * N)

    def call():
        d.api.ops_gemm(d.po, M, N, K, ic.mat(A, 0, K), ic.mat(B, 0, K), 1, ic.mat(out, 0, N), 1, 1,
                       None, 0, None, 0, 1.0, 0, 0.0)
    return call, out, (a.astype(np.float64) @ b.astype(np.float64).T).ravel()


def conv(d, ic, C, K, H, W):
    rng = np.random.default_rng(C + H)
    x = rng.standard_normal((1, C, H, W)).astype(np.float32)
    w = (rng.standard_normal((K, C, 5, 5)) / (25 * C) ** 0.5).astype(np.float32)
    X, Wt, B, out = d.upload(x), d.upload(w), d.zeros(K), d.zeros(K * H * W)
    g = ic.geom(5, 5, 1, 1, 2, 2, 1, 1, 1)

    def call():
        d.api.ops_conv2d_batch(d.po, 1, X.mem, C * H * W, C, H, W, Wt.mem, B.mem, K, ic.C.byref(g),
                               None, None, None, 0, 0.0, out.mem, K * H * W)
    want = F.conv2d(torch.from_numpy(x).double(), torch.from_numpy(w).double(), padding=2)
    return call, out, want.numpy().ravel()


def close(got, want):
    return np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


# 288 tiles of 128 x 128 (32 of them cut) or 1152 of 64 x 64 (none); 512 blocks
# and filters, or 512 blocks and none.
@pytest.mark.parametrize("make,size", [(gemm, (2304, 2000, 1024)), (conv, (32, 64, 256, 256))])
def test_recorded_without_work_memory(make, size, fresh, ic):
    print(f"[graph work] {make.__name__} {size}", flush=True)
    d = fresh
    call, out, want = make(d, ic, *size)
    assert d.ops.scratch_bytes == 0
    d.api.ocl_graph_begin(d.pb)
    call()
    graph = d.api.ocl_graph_end(d.pb)
    try:
        assert d.ops.scratch_bytes == 0
        first = None
        for _ in range(3):
            call()  # eager, which grows the buffer
            assert close(d.read(out), want)
            d.api.ocl_fill(d.pb, out.mem, 0, len(want), 0.0)
            d.finish()
            d.api.ocl_graph_launch(d.pb, graph)
            got = d.read(out)
            first = got if first is None else first
            assert close(got, want) and np.array_equal(got, first)
        assert d.ops.scratch_bytes > 0
        # With the buffer grown, the recording holds the eager call's kernel.
        call()
        eager = d.read(out)
        d.api.ocl_graph_begin(d.pb)
        call()
        ic.lib().ocl_graph_free(graph)
        graph = d.api.ocl_graph_end(d.pb)
        d.api.ocl_fill(d.pb, out.mem, 0, len(want), 0.0)
        d.api.ocl_graph_launch(d.pb, graph)
        assert np.array_equal(d.read(out), eager)
    finally:
        ic.lib().ocl_graph_free(graph)


# Both kernels cut their work into pieces: 64 tiles of 64 x 64; 104 or 208 blocks.
@pytest.mark.parametrize("make,size", [(gemm, (500, 500, 2048)), (conv, (32, 40, 128, 200))])
def test_refused_without_work_memory(make, size, fresh, ic):
    print(f"[graph work] refused {make.__name__} {size}", flush=True)
    d = fresh
    call, out, want = make(d, ic, *size)
    d.api.ocl_graph_begin(d.pb)
    try:
        d.api.ocl_fill(d.pb, out.mem, 0, 4, 0.0)
        with pytest.raises(ic.IcoregError, match="graph is being recorded"):
            call()
    finally:
        ic.lib().ocl_graph_free(d.api.ocl_graph_end(d.pb))
    call()
    assert close(d.read(out), want)
