"""Many-row matmuls on the fp16 GEMM (ggq_gemm_f16.hip): every format and
activation treatment on each of its kernels and tiles (K split over 8
wavefronts with 16 / 32 columns and 16 / 32 / 64 rows a workgroup, the ring
with one, two and four K slices), with ragged rows and columns, fewer and more
superblocks than the wavefronts that share K, a K that is no multiple of 256;
and its per-stream workspace (streams, capture).

Tolerance: an activation row is hi + lo fp16 (2^-23 of each value) and a
product sum of K values is at most 3 K / 16 matrix-core steps and K / 256 + 8
fp32 additions, each within 2^-24 of a partial sum of about the spread of the
result, (sum_k x_k^2 w_k^2)^1/2: errors are taken relative to that spread,
their root mean square below sqrt(3 K / 16 + K / 256 + 8) 2^-24 and 4e-7.
"""
import ctypes

import numpy as np
import pytest

import ggnpu_amd.lib as gl
from tests.gpu_util import dev, host, ptr, stream_handle

pytestmark = pytest.mark.gpu

TYPES = [int(t) for t in gl.GgmlType]
# (N, K, M); the rule for fp32 rows asks for some millions of weights
SHAPES = [(3700, 2304, 9), (8211, 1024, 16), (2050, 2048, 31), (8211, 1024, 32), (1000, 4352, 64), (4130, 1280, 33),
          (515, 4096, 129), (2060, 1280, 300), (600, 8448, 65), (4100, 768, 600), (16500, 512, 520)]
SHAPES32 = [(2800, 1568, 64), (4130, 1568, 50), (2060, 1312, 300), (4100, 800, 600), (16500, 544, 520)]  # 32-value blocks
SMALL = [(1, 256, 9), (33, 512, 31), (130, 1024, 32), (65, 768, 64), (31, 4352, 65), (96, 2304, 129)]  # int8 codes


def tol(K):
    return max(4e-7, np.sqrt(3 * K / 16 + K / 256 + 8) * 2.0 ** -24)


@pytest.fixture(scope="module")
def ctx():
    import torch
    assert torch.cuda.is_available()
    c = gl.Context(0)
    yield c
    c.close()


def weights(t, N, K, seed):
    return gl.encode(t, (np.random.default_rng(seed).standard_normal((N, K)) * 0.02).astype(np.float32))


def rows(M, K, seed):
    """Normal rows; row 1 zero, row 2 tiny, row 3 huge, row 4 with one outlier."""
    a = np.random.default_rng(seed).standard_normal((M, K)).astype(np.float32)
    a[1], a[2], a[3] = 0, a[2] * np.float32(1e-30), a[3] * np.float32(1e30)
    a[4, K // 3] = 300.0
    return a


def check(orc, got, t, raw, N, K, a, act):
    """At most 96 columns (both ends among them) against the oracle."""
    idx = np.arange(N) if N <= 96 else np.unique(np.r_[0:16, N - 40:N, np.random.default_rng(N).choice(N, 40)])
    raw = raw.reshape(N, -1)[idx].reshape(-1)
    ref = orc.mul_mat_f64(t, raw, len(idx), K, a, act)
    w = orc.dequant(t, raw).reshape(len(idx), K).astype(np.float64)
    assert np.isfinite(got).all() and not got[1].any()
    live = [m for m in range(len(a)) if m != 1]
    spread = np.sqrt((a[live].astype(np.float64) ** 2) @ (w ** 2).T)
    err = (got[live][:, idx] - ref[live]) / spread
    assert np.sqrt((err ** 2).mean()) < tol(K)
    assert np.abs(err).max() < 8 * tol(K)


def run(ctx, orc, t, N, K, M, act, i):
    import torch
    raw, a = weights(t, N, K, i), rows(M, K, 50 + i)
    pad, ldc = 1 + i % 3, N + i % 4  # unaligned rows, padded outputs
    x = torch.zeros((M, K + pad), device="cuda")
    x[:, :K].copy_(torch.from_numpy(a))
    y = torch.full((M, ldc), 7.0, device="cuda")
    dW = dev(raw)
    ctx.check(ctx.lib.ggq_mul_mat_dev(ctx.h, ptr(dW), t, N, K, ptr(x), K + pad, ptr(y), ldc, M, act, stream_handle()),
              "mul_mat")
    got = host(y)
    assert (got[:, N:] == 7.0).all()
    check(orc, got[:, :N], t, raw, N, K, a, act)


@pytest.mark.parametrize("act", [0, 1, 2])
@pytest.mark.parametrize("t", TYPES)
def test_tiles_vs_oracle(ctx, orc, t, act):
    for i, s in enumerate(SHAPES32 if gl.BLOCK[gl.GgmlType(t)][0] == 32 else SHAPES):
        run(ctx, orc, t, *s, act, i)


@pytest.mark.parametrize("act", [0, 2])
@pytest.mark.parametrize("t", TYPES)
def test_values_far_below_the_rows_largest(ctx, orc, t, act):
    """Rows whose first superblock is up to 2^60 above the others, against weights
    that are zero there: the others keep their bits (the tolerance is relative
    to their share alone)."""
    import torch
    for i, (N, K, M) in enumerate([(1000, 4352, 64), (600, 8448, 65), (2060, 1280, 300), (4100, 768, 600), (16500, 512, 520)]):
        w = np.random.default_rng(i).standard_normal((N, K)).astype(np.float32) * np.float32(0.02)
        w[:, :256] = 0
        raw, a = gl.encode(t, w), rows(M, K, 70 + i)
        a[5:, :256] *= np.exp2(np.arange(M - 5) % 61).astype(np.float32)[:, None]
        y, dW, x = torch.full((M, N), float("nan"), device="cuda"), dev(raw), torch.from_numpy(a).cuda()
        ctx.check(ctx.lib.ggq_mul_mat_dev(ctx.h, ptr(dW), t, N, K, ptr(x), K, ptr(y), N, M, act, stream_handle()), "mul_mat")
        check(orc, host(y), t, raw, N, K, a, act)


@pytest.mark.parametrize("t", [12, 13, 14, 23])
def test_codes_small_vs_oracle(ctx, orc, t):
    for i, s in enumerate(SMALL):
        run(ctx, orc, t, *s, 1, i)


def test_batches_share_rows(ctx, orc):
    """Entries of one type and of several, sharing their rows or not, in one call."""
    import torch
    M, K = 50, 1024
    a = [rows(M, K, 1), rows(M, K, 2)]
    x = [torch.from_numpy(v).cuda() for v in a]
    spec = [(12, 2070, 0), (12, 33, 0), (14, 1041, 0), (8, 64, 1), (13, 4500, 1), (20, 950, 0)]
    raws = [weights(t, N, K, 9 + i) for i, (t, N, _) in enumerate(spec)]
    ws = [dev(r) for r in raws]
    for act in (0, 1):
        y = [torch.full((M, N), float("nan"), device="cuda") for _, N, _ in spec]
        d = (gl.GemvDesc * len(spec))()
        for i, (t, N, s) in enumerate(spec):
            d[i].W, d[i].type, d[i].N, d[i].K, d[i].A, d[i].C = ws[i].data_ptr(), t, N, K, x[s].data_ptr(), y[i].data_ptr()
        ctx.check(ctx.lib.ggq_mul_mat_batch_act_dev(ctx.h, d, len(spec), M, act, stream_handle()), "batch")
        for i, (t, N, s) in enumerate(spec):
            check(orc, host(y[i]), t, raws[i], N, K, a[s], act)


def call(c, W, t, N, K, x, y, M, stream):
    c.check(c.lib.ggq_mul_mat_dev(c.h, ptr(W), t, N, K, ptr(x), K, ptr(y), N, M, 0, ctypes.c_void_p(stream.cuda_stream)),
            "mul_mat")


def test_streams_do_not_share_planes(orc):
    """fp32 calls queued on ten streams of one context without ordering (more
    streams than the context keeps planes for) all give their own result."""
    import torch
    c = gl.Context(0)
    try:
        t, N, K, M = 12, 2112, 2048, 48
        raw = weights(t, N, K, 3)
        W = dev(raw)
        a = [np.random.default_rng(i).standard_normal((M, K)).astype(np.float32) for i in range(10)]
        x = [torch.from_numpy(v).cuda() for v in a]
        y = [torch.zeros((M, N), device="cuda") for _ in a]
        streams = [torch.cuda.Stream() for _ in a]
        torch.cuda.synchronize()
        for _ in range(5):
            for i, s in enumerate(streams):
                call(c, W, t, N, K, x[i], y[i], M, s)
        torch.cuda.synchronize()
        for i in range(len(a)):
            assert orc.rel_l2(host(y[i])[:, :64], orc.mul_mat_f64(t, raw[: 64 * 1152], 64, K, a[i], 0)) < tol(K)
    finally:
        c.close()


def test_capture_needs_no_reserve_and_keeps_its_planes(orc):
    """An fp32 many-row call is captured on a fresh context (no workspace), and
    after a warm-up with its planes: replays on another stream stay right while
    eager calls run on the stream the graph was captured on."""
    import torch
    c = gl.Context(0)
    try:
        t, N, K, M = 14, 2064, 2048, 40
        raw = weights(t, N, K, 4)
        W = dev(raw)
        rng = np.random.default_rng(8)
        x, y = torch.zeros((M, K), device="cuda"), torch.zeros((M, N), device="cuda")
        a2 = rng.standard_normal((M, K)).astype(np.float32)
        x2, y2 = torch.from_numpy(a2).cuda(), torch.zeros((M, N), device="cuda")
        raw64 = raw[: 64 * 1680]
        ref2 = orc.mul_mat_f64(t, raw64, 64, K, a2, 0)
        s, other = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        for warm in (False, True):
            if warm:
                call(c, W, t, N, K, x, y, M, s)
                torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=s):
                call(c, W, t, N, K, x, y, M, s)
            for _ in range(3):
                a = rng.standard_normal((M, K)).astype(np.float32)
                x.copy_(torch.from_numpy(a))
                y.zero_()
                y2.zero_()
                torch.cuda.synchronize()
                for _ in range(4):
                    with torch.cuda.stream(other):
                        g.replay()
                    call(c, W, t, N, K, x2, y2, M, s)
                torch.cuda.synchronize()
                assert orc.rel_l2(host(y)[:, :64], orc.mul_mat_f64(t, raw64, 64, K, a, 0)) < tol(K)
                assert orc.rel_l2(host(y2)[:, :64], ref2) < tol(K)
    finally:
        c.close()
