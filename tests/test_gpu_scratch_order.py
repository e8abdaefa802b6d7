"""GPU test of the shared scratch's ordering between the context's own stream and others: calls
that quantize into it, enqueued back to back on alternating streams, give the results of the
same calls one at a time."""
import time

import pytest

from aikit_amd import enchip, workloads

pytestmark = pytest.mark.gpu


def test_alternating_streams_share_the_scratch():
    import torch

    g = workloads.rng(31)
    M, K, N = 3000, 1024, 1024  # two kernels a call: the quantizer writes the scratch, the GEMM reads it
    with enchip.Context(0) as c:
        w = c.register_weight(*workloads.int8_weights(g, N, K))
        a = [torch.from_numpy(workloads.activations(g, M, K)).cuda() for _ in range(12)]
        out, want = ([torch.empty((M, N), device="cuda") for _ in a] for _ in range(2))
        torch.cuda.synchronize()
        for x, y in zip(a, want):
            c.linear_dev(w, x.data_ptr(), M, 0, enchip.ACT_NONE, y.data_ptr())
            torch.cuda.synchronize()
        others = [torch.cuda.Stream(), torch.cuda.Stream()]
        order = [0, 1, 0, 0, 2, 1, 0, 2, 2, 0, 0, 1]  # 0: the context's stream
        for rep in range(5):
            for x, y, o in zip(a, out, order):
                c.linear_dev(w, x.data_ptr(), M, 0, enchip.ACT_NONE, y.data_ptr(), 0 if o == 0 else others[o - 1].cuda_stream)
        del others[1]  # a caller's stream may go before the scratch is used again
        c.linear_dev(w, a[0].data_ptr(), M, 0, enchip.ACT_NONE, out[0].data_ptr())
        torch.cuda.synchronize()
        for y, z in zip(out, want):
            assert torch.equal(y.view(torch.int32), z.view(torch.int32))


def test_another_stream_waits_for_the_scratch_alone():
    # The context's stream: a linear (it uses the scratch), then f32 products of some 100 ms (they do
    # not). A linear on another stream, once such a stream has used the scratch before, waits for the
    # first linear and not for the products.
    import torch

    g = workloads.rng(32)
    M, K, N = 512, 768, 768
    with enchip.Context(0) as c:
        w = c.register_weight(*workloads.int8_weights(g, N, K))
        a = torch.from_numpy(workloads.activations(g, M, K)).cuda()
        big = torch.randn((8192, 8192), device="cuda")
        out, prod = torch.empty((M, N), device="cuda"), torch.empty((8192, 8192), device="cuda")
        s = torch.cuda.Stream()
        torch.cuda.synchronize()

        def linear(stream):
            c.linear_dev(w, a.data_ptr(), M, 0, enchip.ACT_NONE, out.data_ptr(), stream)

        def products(n):
            for _ in range(n):
                c.matmul_bt_f32_dev(big.data_ptr(), 8192, big.data_ptr(), 8192, enchip.B_NK, prod.data_ptr(), 8192, 8192,
                                    8192, 8192)

        linear(0), products(1), linear(s.cuda_stream)  # kernels loaded, the other stream known
        torch.cuda.synchronize()
        print("[case] scratch order beside f32 products", flush=True)
        linear(0), products(30), linear(s.cuda_stream)
        t0 = time.perf_counter()
        s.synchronize()
        t1 = time.perf_counter()
        torch.cuda.synchronize()
        t2 = time.perf_counter()
        assert t1 - t0 < (t2 - t0) / 4, f"the other stream ended after {t1 - t0:.4f} of {t2 - t0:.4f} s"
