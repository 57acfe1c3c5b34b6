"""Workspace contract of the device entry points (include/ggq.h): a call being
captured into a HIP graph never allocates (it fails with a clear message
when its workspace is too small), ggq_reserve sizes the workspace ahead of a
capture, and a graph captured before the workspace grows stays valid after
the growth (outgrown buffers are kept until ggq_destroy)."""
import ctypes

import numpy as np
import pytest

import ggnpu_amd.lib as gl
from tests import test_gpu_parity as t
from tests.gpu_util import dev, host, ptr

pytestmark = pytest.mark.gpu


def q8_call(c, dW, N, K, x, y, M, stream):
    return c.lib.ggq_mul_mat_dev(c.h, ctypes.c_void_p(dW.data_ptr()), 8, N, K, ctypes.c_void_p(x.data_ptr()), K,
                                 ctypes.c_void_p(y.data_ptr()), N, M, int(gl.ActMode.Q8_ROW), stream)


def test_capture_refuses_growth_then_reserve(orc):
    import torch
    c = gl.Context(0)
    try:
        N, K, M = 512, 4096, 64  # K > 2048: quantized into the workspace, split-K partials
        raw = t.weights(8, N, K, seed=3)
        dW = dev(raw)
        A = np.random.default_rng(3).standard_normal((M, K)).astype(np.float32)
        x = torch.from_numpy(A).cuda()
        y = torch.zeros((M, N), device="cuda")
        s = torch.cuda.Stream()
        sh = ctypes.c_void_p(s.cuda_stream)
        torch.cuda.synchronize()
        # fresh context: no workspace yet, so the captured call is refused
        g = torch.cuda.CUDAGraph()
        with torch.cuda.stream(s):
            with torch.cuda.graph(g, stream=s):
                st = q8_call(c, dW, N, K, x, y, M, sh)
        assert st == int(gl.Status.ERROR)
        assert b"captured" in c.lib.ggq_last_error_message(c.h)
        del g
        torch.cuda.synchronize()
        # reserve, then the same capture works and replays match the oracle
        c.check(c.lib.ggq_reserve(c.h, 64 << 20), "reserve")
        g = torch.cuda.CUDAGraph()
        with torch.cuda.stream(s):
            with torch.cuda.graph(g, stream=s):
                c.check(q8_call(c, dW, N, K, x, y, M, sh), "captured q8")
        ref = orc.mul_mat_f64(8, raw, N, K, A, 1)
        for _ in range(3):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert orc.rel_l2(y.cpu().numpy(), ref) < t.TOL
    finally:
        c.close()


def test_graph_survives_workspace_growth(orc):
    """Capture with a small workspace, grow it with a larger eager call, then
    replay: the graph still reads the (kept) old buffer and is correct."""
    import torch
    c = gl.Context(0)
    try:
        N, K = 384, 4096  # the workspace path (K > 2048)
        raw = t.weights(8, N, K, seed=4)
        dW = dev(raw)
        rng = np.random.default_rng(4)
        A1 = rng.standard_normal((16, K)).astype(np.float32)
        A2 = rng.standard_normal((256, K)).astype(np.float32)
        x1, x2 = torch.from_numpy(A1).cuda(), torch.from_numpy(A2).cuda()
        y1, y2 = torch.zeros((16, N), device="cuda"), torch.zeros((256, N), device="cuda")
        s = torch.cuda.Stream()
        sh = ctypes.c_void_p(s.cuda_stream)
        with torch.cuda.stream(s):
            c.check(q8_call(c, dW, N, K, x1, y1, 16, sh), "warm-up")
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.stream(s):
            with torch.cuda.graph(g, stream=s):
                c.check(q8_call(c, dW, N, K, x1, y1, 16, sh), "captured")
        with torch.cuda.stream(s):
            c.check(q8_call(c, dW, N, K, x2, y2, 256, sh), "growing call")
        torch.cuda.synchronize()
        assert orc.rel_l2(y2.cpu().numpy(), orc.mul_mat_f64(8, raw, N, K, A2, 1)) < t.TOL
        ref1 = orc.mul_mat_f64(8, raw, N, K, A1, 1)
        for _ in range(3):
            y1.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert orc.rel_l2(y1.cpu().numpy(), ref1) < t.TOL
    finally:
        c.close()


def test_capture_needs_no_workspace_on_the_panel_gemm(orc):
    """K <= 2048: the prefill GEMM quantizes the rows inside its own launch
    and uses no workspace, so a fresh context captures it without
    ggq_reserve; replays on fresh inputs match the oracle."""
    import torch
    c = gl.Context(0)
    try:
        N, K, M = 640, 1536, 96
        raw = t.weights(8, N, K, seed=5)
        dW = dev(raw)
        rng = np.random.default_rng(5)
        x = torch.zeros((M, K), device="cuda")
        y = torch.zeros((M, N), device="cuda")
        s = torch.cuda.Stream()
        sh = ctypes.c_void_p(s.cuda_stream)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.stream(s):
            with torch.cuda.graph(g, stream=s):
                c.check(q8_call(c, dW, N, K, x, y, M, sh), "captured panel GEMM")
        for _ in range(3):
            A = rng.standard_normal((M, K)).astype(np.float32)
            x.copy_(torch.from_numpy(A))
            y.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert orc.rel_l2(y.cpu().numpy(), orc.mul_mat_f64(8, raw, N, K, A, 1)) < t.TOL
    finally:
        c.close()


def capture(g, s, work):
    """torch.cuda.graph without its synchronizations: work queued on `s` may still run."""
    import torch
    with torch.cuda.stream(s):
        g.capture_begin()
        work()
        g.capture_end()


def f32_call(c, t_, W, N, K, x, y, M, s):
    c.check(c.lib.ggq_mul_mat_dev(c.h, ctypes.c_void_p(W.data_ptr()), t_, N, K, ctypes.c_void_p(x.data_ptr()), K,
                                  ctypes.c_void_p(y.data_ptr()), N, M, 0, ctypes.c_void_p(s.cuda_stream)), "mul_mat")


@pytest.mark.parametrize("N,K,M", [(2064, 2048, 40), (2064, 4352, 16)])
def test_capture_beside_queued_eager_calls(orc, N, K, M):
    """fp32 many-row calls (planes; the slices' sums of few rows) queued on a
    stream before a capture on it still run while the graph replays on another
    stream: neither disturbs the other, bit for bit."""
    import torch
    c = gl.Context(0)
    try:
        raw = t.weights(14, N, K, seed=6)
        W = dev(raw)
        x = [torch.randn((M, K), device="cuda") for _ in range(2)]
        y = [torch.zeros((M, N), device="cuda") for _ in range(17)]
        s, other = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        want = []
        for a in x:
            f32_call(c, 14, W, N, K, a, y[0], M, s)
            torch.cuda.synchronize()
            want.append(y[0].clone())
        assert orc.rel_l2(host(want[0])[:, :64], orc.mul_mat_f64(14, raw[: 64 * (K // 256) * 210], 64, K, host(x[0]), 0)) < t.TOL
        for _ in range(3):
            for v in y:
                v.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(s):
                torch.cuda._sleep(5_000_000)
            for i in range(16):
                f32_call(c, 14, W, N, K, x[0], y[i], M, s)
            g = torch.cuda.CUDAGraph()
            capture(g, s, lambda: [f32_call(c, 14, W, N, K, x[1], y[16], M, s) for _ in range(16)])
            with torch.cuda.stream(other):
                for _ in range(8):
                    g.replay()
            torch.cuda.synchronize()
            for i in range(16):
                assert torch.equal(y[i], want[0]), i
            assert torch.equal(y[16], want[1])
    finally:
        c.close()


# (type, M, K): Q6_K rows and long rows of Q4_K use the int8 GEMM's workspace without planes
@pytest.mark.parametrize("entry", ["row", "codes", "batch"])
@pytest.mark.parametrize("ty,M,K", [(14, 40, 2048), (12, 16, 4352)])
def test_one_warm_up_prepares_every_capture(orc, ty, M, K, entry):
    """int8 rows: after one eager call, any number of captures on another stream
    are accepted; those with planes equal the eager call bit for bit, the ones
    beyond what was set aside agree with the oracle."""
    import torch
    N, captures = 528, 12
    c = gl.Context(0)
    try:
        raw = t.weights(ty, N, K, seed=ty)
        W = dev(raw)
        a = np.random.default_rng(K).standard_normal((M, K)).astype(np.float32)
        x, y = torch.from_numpy(a).cuda(), torch.zeros((M, N), device="cuda")
        q, sa = torch.zeros((M, K), dtype=torch.int8, device="cuda"), torch.zeros(M, device="cuda")
        c.check(c.lib.ggq_quantize_act_dev(c.h, ptr(x), K, M, K, 1, ptr(q), ptr(sa), None), "quantize")
        d = (gl.GemvDesc * 1)()
        d[0].W, d[0].type, d[0].N, d[0].K, d[0].A, d[0].C = W.data_ptr(), ty, N, K, x.data_ptr(), y.data_ptr()

        def call(s):
            h = ctypes.c_void_p(s.cuda_stream)
            if entry == "row":
                return c.lib.ggq_mul_mat_dev(c.h, ptr(W), ty, N, K, ptr(x), K, ptr(y), N, M, 1, h)
            if entry == "codes":
                return c.lib.ggq_mul_mat_q8_dev(c.h, ptr(W), ty, N, K, ptr(q), ptr(sa), M, ptr(y), N, h)
            return c.lib.ggq_mul_mat_batch_act_dev(c.h, d, 1, M, 1, h)
        warm, s = torch.cuda.Stream(), torch.cuda.Stream()
        torch.cuda.synchronize()
        c.check(call(warm), "warm-up")
        torch.cuda.synchronize()
        want = y.clone()
        ref = orc.mul_mat_f64(ty, raw, N, K, a, 1)
        status, graphs = [], []
        for _ in range(captures):
            g = torch.cuda.CUDAGraph()
            capture(g, s, lambda: status.append(call(s)))
            graphs.append(g)
        assert status == [0] * captures
        for i, g in enumerate(graphs):
            for _ in range(2):
                y.zero_()
                g.replay()
                torch.cuda.synchronize()
                assert orc.rel_l2(host(y), ref) < t.TOL
                if i < 8:
                    assert torch.equal(y, want), i
    finally:
        c.close()


def test_reserve_prepares_captures_of_many_rows(orc):
    """After ggq_reserve alone a capture records what an eager call runs."""
    import torch
    N, K, M = 2064, 2048, 40
    c = gl.Context(0)
    try:
        W = dev(t.weights(14, N, K, seed=1))
        x, y, want = torch.randn((M, K), device="cuda"), torch.zeros((M, N), device="cuda"), torch.zeros((M, N), device="cuda")
        s = torch.cuda.Stream()
        c.check(c.lib.ggq_reserve(c.h, 4 << 20), "reserve")
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        capture(g, s, lambda: f32_call(c, 14, W, N, K, x, y, M, s))
        f32_call(c, 14, W, N, K, x, want, M, s)
        for _ in range(3):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, want)
    finally:
        c.close()


@pytest.mark.parametrize("N,K,M", [(2064, 2048, 40), (2064, 4352, 16)])
def test_every_stream_runs_the_same_kernels(N, K, M):
    """Unordered fp32 many-row calls on more streams than a context keeps buffers
    for, hipStreamPerThread among them, each give the first stream's result bit
    for bit, also while earlier calls on other streams still run."""
    import torch
    c = gl.Context(0)
    try:
        W = dev(t.weights(14, N, K, seed=2))
        streams = [torch.cuda.Stream().cuda_stream for _ in range(20)] + [2]
        x = [torch.randn((M, K), device="cuda") for _ in streams]
        y = [torch.zeros((M, N), device="cuda") for _ in streams]
        want = [torch.zeros((M, N), device="cuda") for _ in streams]
        torch.cuda.synchronize()

        def call(a, out, s):
            c.check(c.lib.ggq_mul_mat_dev(c.h, ptr(W), 14, N, K, ptr(a), K, ptr(out), N, M, 0, ctypes.c_void_p(s)), "mul_mat")
        for a, out in zip(x, want):
            call(a, out, streams[0])
        torch.cuda.synchronize()
        for _ in range(3):
            for v in y:
                v.zero_()
            torch.cuda.synchronize()
            with torch.cuda.stream(torch.cuda.ExternalStream(streams[9])):
                torch.cuda._sleep(2_000_000)
            for _ in range(4):
                for a, out, s in zip(x, y, streams):
                    call(a, out, s)
            torch.cuda.synchronize()
            for i, (out, ref) in enumerate(zip(y, want)):
                assert torch.equal(out, ref), i
    finally:
        c.close()


# (type, K, M, bytes reserved): the activation-panel GEMM (K <= 2048, no workspace), then the int8 GEMM, whose
# workspace is reserved with less than the planes would take
@pytest.mark.parametrize("ty,K,M,reserve", [(12, 2048, 100, 0), (13, 1792, 33, 0), (23, 1792, 100, 0),
                                            (14, 2048, 100, 500_000), (14, 4352, 33, 1 << 20), (12, 4352, 100, 1 << 20),
                                            (13, 4352, 33, 1 << 20), (23, 4352, 20, 1 << 20)])
def test_int8_kernels_without_planes(orc, ty, K, M, reserve):
    """What captures of int8 rows record when no planes are set aside, through
    each entry point: against the oracle, fp32 rows and codes bit for bit alike."""
    import torch
    N = 72
    c = gl.Context(0)
    try:
        raw = t.weights(ty, N, K, seed=K + ty)
        W = dev(raw)
        a = np.random.default_rng(K + M).standard_normal((M, K)).astype(np.float32)
        x, y = torch.from_numpy(a).cuda(), [torch.zeros((M, N), device="cuda") for _ in range(6)]
        q, sa = torch.zeros((M, K), dtype=torch.int8, device="cuda"), torch.zeros(M, device="cuda")
        c.check(c.lib.ggq_quantize_act_dev(c.h, ptr(x), K, M, K, 1, ptr(q), ptr(sa), None), "quantize")
        c.check(c.lib.ggq_reserve(c.h, reserve), "reserve")
        gd, bd = (gl.GemmDesc * 2)(), (gl.GemvDesc * 2)()
        for i in range(2):
            gd[i].W, gd[i].N, gd[i].C, gd[i].ldc = W.data_ptr(), N, y[2 + i].data_ptr(), N
            bd[i].W, bd[i].type, bd[i].N, bd[i].K = W.data_ptr(), ty, N, K
            bd[i].A, bd[i].C = x.data_ptr(), y[4 + i].data_ptr()
        s = torch.cuda.Stream()
        h = ctypes.c_void_p(s.cuda_stream)
        status = []
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        capture(g, s, lambda: status.extend([
            c.lib.ggq_mul_mat_dev(c.h, ptr(W), ty, N, K, ptr(x), K, ptr(y[0]), N, M, 1, h),
            c.lib.ggq_mul_mat_q8_dev(c.h, ptr(W), ty, N, K, ptr(q), ptr(sa), M, ptr(y[1]), N, h),
            c.lib.ggq_mul_mat_q8_batch_dev(c.h, gd, 2, ty, K, ptr(q), ptr(sa), M, h),
            c.lib.ggq_mul_mat_batch_act_dev(c.h, bd, 2, M, 1, h)]))
        assert status == [0] * 4, c.lib.ggq_last_error_message(c.h)
        ref = orc.mul_mat_f64(ty, raw, N, K, a, 1)
        for _ in range(2):
            for v in y:
                v.zero_()
            g.replay()
            torch.cuda.synchronize()
            for v in y:
                assert orc.rel_l2(host(v), ref) < t.TOL
            assert torch.equal(y[0], y[1])
    finally:
        c.close()
