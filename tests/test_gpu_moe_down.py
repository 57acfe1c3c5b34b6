"""MoE layers of a few tokens, where one launch does the SwiGLU, the routed and
shared down projections and the weighted sum: every format, rows of 1 to 64
pieces (and one more, which the separate launches take), more experts a token
than wavefronts, with and without a shared expert; every stage of every expert
(the traced SwiGLU and down rows are the launch's own) at the other paths' bar.
"""
import pytest

from tests.test_gpu_moe_stages import check_stages, ctx, run_layer  # noqa: F401

pytestmark = pytest.mark.gpu

CASES = [(1, 512, 256, 8, 4), (8, 512, 256, 8, 4), (2, 1280, 512, 16, 6), (1, 256, 1024, 4, 2), (1, 256, 2048, 3, 2),
         (1, 256, 2304, 3, 2), (1, 256, 256, 40, 33)]  # T, H, F, E, k
CASES32 = [(1, 288, 32, 8, 4), (3, 544, 288, 8, 4), (2, 256, 1056, 4, 2)]


@pytest.mark.parametrize("t", [8, 12, 13, 14, 20, 23])
def test_few_tokens(ctx, orc, t):  # noqa: F811
    for i, (T, H, F, E, k) in enumerate(CASES + (CASES32 if t in (8, 20) else [])):
        types = (t if t in (8, 20) else 12, t if t in (8, 20) else 12, t)
        L = run_layer(ctx, T, H, F, E, k, types, 0, seed=t + i, shared=i % 2 == 0)
        check_stages(orc, L, T, H, F, E, k, types, 0)
