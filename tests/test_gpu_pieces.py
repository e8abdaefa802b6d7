"""GPU parity of the W8A8 GEMM in pieces (a few hundred to a few thousand rows): outputs and
int32 accumulators bit for bit against the CPU oracle, at the edges of its piece sizes."""
import numpy as np
import pytest

import oracle
from aikit_amd import enchip, workloads

pytestmark = pytest.mark.gpu

# (M, K, N, piece): one row past the small-M kernels, one 32-column group and less, fewer K
# stages than wavefronts (K = 64: three have none; 192, 320: an odd number), a remainder in
# every dimension, N not a multiple of 4, and each piece size with its last pieces cut off
SHAPES = [(33, 64, 4, "32, 32"), (33, 64, 1, "32, 32"), (64, 128, 36, "32, 32"), (65, 192, 1000, "32, 32"),
          (300, 3072, 768, "32, 32"), (511, 768, 2300, "64, 32"), (97, 320, 8003, "64, 32"), (1025, 768, 1001, "64, 32"),
          (1000, 1536, 1028, "64, 64"), (513, 4096, 1999, "64, 64"), (333, 1001, 257, "32, 32")]


def bits(x):
    return np.ascontiguousarray(x, np.float32).view(np.uint32)


@pytest.mark.parametrize("M,K,N,piece", SHAPES)
def test_pieces_match_oracle(ctx, M, K, N, piece):
    g = workloads.rng(1201 + M + K + N)
    a = workloads.activations(g, M, K)
    a[M // 2] = 0  # an all-zero row: scale 0
    wq, ws = workloads.int8_weights(g, N, K)
    ws *= np.float32(0.002)  # pre-activations on every branch of the GELU, most on its series
    b = workloads.bias(g, N)
    w = ctx.register_weight(wq, ws)
    try:
        name = ctx.gemm_kernel_name(w, M, enchip.ACT_NONE)
        print(f"[case] pieces M={M} K={K} N={N} via {name} / {ctx.gemm_kernel_name(w, M, enchip.ACT_GELU)}", flush=True)
        if ctx.device_info()["num_cus"] == 256:
            assert piece in name, name
        plain, acc = ctx.linear(w, a, bias=b, act=enchip.ACT_NONE, want_acc=True)
        nobias = ctx.linear(w, a)
        gelu = ctx.linear(w, a, bias=b, act=enchip.ACT_GELU)
    finally:
        ctx.release_weight(w)
    aq, _ = oracle.quantize_activations(a, M, K)
    assert np.array_equal(acc, oracle.acc_i32(aq, wq, M, K, N))
    assert np.array_equal(bits(plain), bits(oracle.w8a8_linear(a, wq, ws, b, 0, M, K, N)))
    assert np.array_equal(bits(nobias), bits(oracle.w8a8_linear(a, wq, ws, None, 0, M, K, N)))
    assert np.array_equal(bits(gelu), bits(oracle.w8a8_linear(a, wq, ws, b, 1, M, K, N)))
