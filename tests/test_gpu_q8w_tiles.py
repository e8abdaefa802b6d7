"""GPU tests of the weight-only int8 product's tiles at their edges: exact on integers (every
product and partial sum below 2^24, so f32 is exact in any order)."""
import numpy as np
import pytest

from aikit_amd import workloads

pytestmark = pytest.mark.gpu


# (M, K, N): one 32 x 32 tile per CU at most; 32 x 128 tiles, 128-deep chunks (a padded K that
# is an odd number of 64s: the last chunk half past it) and 64-deep ones; 128 x 256 tiles (256
# of them, and more); K not a multiple of 4 (values loaded one by one); one row, one channel
@pytest.mark.parametrize("M,K,N", [(33, 200, 250), (700, 320, 700), (513, 321, 1001), (1000, 70, 1300), (1500, 193, 3001),
                                   (4090, 96, 2040), (7000, 33, 3001), (1, 1000, 9000), (9001, 64, 1)])
def test_tiles_exact_on_integers(ctx, M, K, N):
    import torch

    g = workloads.rng(400 + M + K + N)
    ai = g.integers(-16, 17, size=(M, K)).astype(np.int8)
    qi = g.integers(-128, 128, size=(N, K)).astype(np.int8)
    s = np.ldexp(1.0, g.integers(-3, 3, size=N)).astype(np.float32)
    print(f"[case] q8w tiles M={M} K={K} N={N}", flush=True)
    w = ctx.register_weight(qi, s)
    try:
        got = ctx.matmul_bt_q8(w, ai.astype(np.float32))
    finally:
        ctx.release_weight(w)
    want = torch.from_numpy(ai).cuda().double() @ torch.from_numpy(qi).cuda().double().t().contiguous()
    want = want.float().cpu().numpy() * s
    assert np.array_equal(got, want)
