"""Matmuls of 5..32 fp32 rows kept in registers (ggq_gemm_rows.hip): every
format with one and two row tiles, fewer and more columns than the workgroups,
K below a superblock's multiple, K split over one, two and five slices with a
short last one, batches of mixed formats, and capture.

Tolerance: a row's superblock is hi + lo fp16 (2^-22 of its largest value), a
product sum of K values is at most 3 K / 32 matrix-core steps and K / 256 + 8
fp32 additions, each within 2^-24 of a partial sum of about the spread of the
result, (sum_k x_k^2 w_k^2)^1/2: the bound of test_gpu_gemm_f16 holds.
"""
import numpy as np
import pytest

import ggnpu_amd.lib as gl
from tests.gpu_util import dev, host, ptr, stream_handle
from tests.test_gpu_gemm_f16 import TYPES, call, check, rows, run, tol, weights

pytestmark = pytest.mark.gpu

# (N, K, M) the rule takes; 32-value blocks from more weights
SHAPES = [(8200, 1024, 6), (4111, 2304, 6), (8200, 1024, 8), (3100, 1024, 9), (1300, 2560, 16), (400, 8448, 12),
          (8209, 1024, 17), (1030, 8192, 31), (4100, 2304, 32), (34000, 256, 32)]
SHAPES32 = [(16400, 1056, 16), (5400, 3136, 9), (16400, 1024, 32), (2100, 8224, 20)]


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    c = gl.Context(0)
    yield c
    c.close()


def run_aligned(ctx, orc, t, N, K, M, i):
    import torch
    raw, a = weights(t, N, K, i), rows(M, K, 50 + i)
    lda, ldc = K + 4 * (i % 3), N + i % 4
    x = torch.full((M, lda), float("nan"), device="cuda")
    x[:, :K].copy_(torch.from_numpy(a))
    y = torch.full((M, ldc), 7.0, device="cuda")
    dW = dev(raw)
    ctx.check(ctx.lib.ggq_mul_mat_dev(ctx.h, ptr(dW), t, N, K, ptr(x), lda, ptr(y), ldc, M, 0, stream_handle()), "mul_mat")
    got = host(y)
    assert (got[:, N:] == 7.0).all()
    check(orc, got[:, :N], t, raw, N, K, a, 0)


@pytest.mark.parametrize("t", TYPES)
def test_rows_vs_oracle(ctx, orc, t):
    shapes = SHAPES32 if gl.BLOCK[gl.GgmlType(t)][0] == 32 else SHAPES
    for i, s in enumerate(shapes):
        run_aligned(ctx, orc, t, *s, i)
    run(ctx, orc, t, *shapes[0], 0, 1)  # rows that are not 16-byte aligned: the other kernels
    run(ctx, orc, t, *shapes[1], 2, 2)  # per-32 int8 rows


@pytest.mark.parametrize("M,K", [(8, 2048), (32, 1024), (20, 4352)])
def test_formats_share_a_launch(ctx, orc, M, K):
    import torch
    a = [rows(M, K, 1), rows(M, K, 2)]
    x = [torch.from_numpy(v).cuda() for v in a]
    spec = [(12, 3070, 0), (14, 1041, 0), (23, 450, 0), (8, 64, 0), (13, 15, 0), (12, 8200, 1)]
    raws = [weights(t, N, K, 9 + i) for i, (t, N, _) in enumerate(spec)]
    ws = [dev(r) for r in raws]
    y = [torch.full((M, N), float("nan"), device="cuda") for _, N, _ in spec]
    d = (gl.GemvDesc * len(spec))()
    for i, (t, N, s) in enumerate(spec):
        d[i].W, d[i].type, d[i].N, d[i].K, d[i].A, d[i].C = ws[i].data_ptr(), t, N, K, x[s].data_ptr(), y[i].data_ptr()
    ctx.check(ctx.lib.ggq_mul_mat_batch_rows_dev(ctx.h, d, len(spec), M, stream_handle()), "batch")
    for i, (t, N, s) in enumerate(spec):
        check(orc, host(y[i]), t, raws[i], N, K, a[s], 0)


@pytest.mark.parametrize("N,K,M", [(8208, 2048, 8), (2064, 4352, 16)])
def test_capture(orc, N, K, M):
    """On a fresh context and after a call on the stream (with the slices' sums)."""
    import torch
    c = gl.Context(0)
    try:
        t = 14
        raw = weights(t, N, K, 4)
        W, raw64 = dev(raw), raw.reshape(N, -1)[:64].reshape(-1)
        x, y = torch.zeros((M, K), device="cuda"), torch.zeros((M, N), device="cuda")
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        for warm in (False, True):
            if warm:
                call(c, W, t, N, K, x, y, M, s)
                torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                call(c, W, t, N, K, x, y, M, s)
            for i in range(3):
                a = np.random.default_rng(i).standard_normal((M, K)).astype(np.float32)
                x.copy_(torch.from_numpy(a))
                y.zero_()
                torch.cuda.synchronize()
                g.replay()
                g.replay()
                torch.cuda.synchronize()
                assert orc.rel_l2(host(y)[:, :64], orc.mul_mat_f64(t, raw64, 64, K, a, 0)) < tol(K)
    finally:
        c.close()
