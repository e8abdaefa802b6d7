"""GPU test of the shared scratch's ordering between the context's own stream and others: calls
that quantize into it, enqueued back to back on alternating streams, give the results of the
same calls one at a time."""
import ctypes
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
        c.linear_dev(w, a[0].data_ptr(), M, 0, enchip.ACT_NONE, out[0].data_ptr())
        torch.cuda.synchronize()
        for y, z in zip(out, want):
            assert torch.equal(y.view(torch.int32), z.view(torch.int32))


def hip():
    """The HIP runtime this process has loaded."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))


@pytest.mark.parametrize("first", [True, False])
def test_a_stream_that_is_gone_was_the_last_user(first):
    # A caller's stream uses the scratch last and is destroyed before the context's stream uses it
    # again: before any use on the context's stream, or after one.
    import torch

    g = workloads.rng(33)
    M, K, N = 3000, 1024, 1024
    with enchip.Context(0) as c:
        w = c.register_weight(*workloads.int8_weights(g, N, K))
        a = [torch.from_numpy(workloads.activations(g, M, K)).cuda() for _ in range(3)]
        out, want = ([torch.empty((M, N), device="cuda") for _ in a] for _ in range(2))
        torch.cuda.synchronize()
        with enchip.Context(0) as alone:
            w1 = alone.register_weight(*workloads.int8_weights(workloads.rng(33), N, K))
            for x, y in zip(a, want):
                alone.linear_dev(w1, x.data_ptr(), M, 0, enchip.ACT_NONE, y.data_ptr())
                torch.cuda.synchronize()
        lib, s = hip(), ctypes.c_void_p()
        for rep in range(5):
            if not first:
                c.linear_dev(w, a[0].data_ptr(), M, 0, enchip.ACT_NONE, out[0].data_ptr())
            assert lib.hipStreamCreate(ctypes.byref(s)) == 0
            print(f"[case] scratch and a destroyed stream, first={first} rep={rep}", flush=True)
            c.linear_dev(w, a[1].data_ptr(), M, 0, enchip.ACT_NONE, out[1].data_ptr(), s.value)
            assert lib.hipStreamDestroy(s) == 0
            c.linear_dev(w, a[2].data_ptr(), M, 0, enchip.ACT_NONE, out[2].data_ptr())
            torch.cuda.synchronize()
            for i in range(int(first), 3):
                assert torch.equal(out[i].view(torch.int32), want[i].view(torch.int32))


@pytest.mark.parametrize("shared", [False, True])
def test_the_scratch_grows_while_in_use(shared):
    # Work on the context's stream (with no event, or with one where another stream has used the
    # scratch) reads the scratch when a call with more rows replaces it.
    import torch

    g = workloads.rng(34)
    K, N = 1024, 1024
    Ms = [2000, 6000, 14000]
    a = [torch.from_numpy(workloads.activations(g, M, K)).cuda() for M in Ms]
    wq, ws = workloads.int8_weights(g, N, K)
    got = []
    for wait in (True, False):
        with enchip.Context(0) as c:
            w = c.register_weight(wq, ws)
            outs = [torch.empty((M, N), device="cuda") for M in Ms]
            s = torch.cuda.Stream()
            torch.cuda.synchronize()
            print(f"[case] scratch growth shared={shared} wait={wait}", flush=True)
            if shared:
                for stream in (0, s.cuda_stream):
                    c.linear_dev(w, a[0].data_ptr(), 100, 0, enchip.ACT_NONE, outs[0].data_ptr(), stream)
                torch.cuda.synchronize()
            for M, x, y in zip(Ms, a, outs):
                c.linear_dev(w, x.data_ptr(), M, 0, enchip.ACT_NONE, y.data_ptr())
                if wait:
                    torch.cuda.synchronize()
            torch.cuda.synchronize()
            got.append(outs)
    for x, y in zip(*got):
        assert torch.equal(x.view(torch.int32), y.view(torch.int32))


def test_another_stream_waits_for_the_scratch_alone():
    # The context's stream: a linear (it uses the scratch), then f32 products of some 100 ms (they do
    # not). A linear on another stream, once such a stream has used the scratch before, waits for the
    # first linear and not for the products. (Streams share a few hardware queues, and work on one
    # queue runs in order: of several streams, one that has a queue of its own shows it.)
    import torch

    g = workloads.rng(32)
    M, K, N = 512, 768, 768
    with enchip.Context(0) as c:
        w = c.register_weight(*workloads.int8_weights(g, N, K))
        a = torch.from_numpy(workloads.activations(g, M, K)).cuda()
        big = torch.randn((8192, 8192), device="cuda")
        out, prod = torch.empty((M, N), device="cuda"), torch.empty((8192, 8192), device="cuda")
        torch.cuda.synchronize()

        def linear(stream):
            c.linear_dev(w, a.data_ptr(), M, 0, enchip.ACT_NONE, out.data_ptr(), stream)

        def products(n):
            for _ in range(n):
                c.matmul_bt_f32_dev(big.data_ptr(), 8192, big.data_ptr(), 8192, enchip.B_NK, prod.data_ptr(), 8192, 8192,
                                    8192, 8192)

        linear(0), products(1)  # kernels loaded
        torch.cuda.synchronize()
        shares = []
        for i in range(8):
            s = torch.cuda.Stream()
            linear(0), linear(s.cuda_stream)  # such a stream has used the scratch
            torch.cuda.synchronize()
            print(f"[case] scratch order beside f32 products, stream {i}", flush=True)
            linear(0), products(30), linear(s.cuda_stream)
            t0 = time.perf_counter()
            s.synchronize()
            t1 = time.perf_counter()
            torch.cuda.synchronize()
            shares.append((t1 - t0) / (time.perf_counter() - t0))
            if shares[-1] < 0.25:
                return
        raise AssertionError(f"the other streams waited for {shares} of the products")
