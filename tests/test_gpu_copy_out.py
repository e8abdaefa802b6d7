"""GPU tests of the staged copy of results to host memory at the edges of its slices (512 KiB),
halves (2 MiB) and launches: every byte, from several threads and contexts."""
import inspect
import os
import subprocess
import sys
import threading

import numpy as np
import pytest

from aikit_amd import enchip, workloads

pytestmark = pytest.mark.gpu

KIB = 1024


# bytes of the codes (one a value): below the staged size, at it, one slice and a tail that is
# not a multiple of 16, a half exactly, a byte past it, two halves and a byte (a third launch
# into the first half), several rounds of both halves
@pytest.mark.parametrize("n", [1024 * KIB - 1, 1024 * KIB, 1536 * KIB + 13, 2048 * KIB, 2048 * KIB + 1, 4096 * KIB + 1,
                               4608 * KIB, 11 * 1024 * KIB + 7])
def test_every_byte_arrives(ctx, n):
    g = workloads.rng(n)
    K = next(k for k in range(4096, 0, -1) if n % k == 0)
    M = n // K
    a = g.integers(-127, 128, size=(M, K)).astype(np.float32)
    a[:, 0] = 127  # scale 1: the codes are the values
    print(f"[case] copy out n={n} M={M} K={K}", flush=True)
    for _ in range(3):  # other values: the staging holds the last call's
        codes, scales = ctx.quant_rows(a)
        assert np.array_equal(codes, a.astype(np.int8))
        assert (scales == 1).all()
        a[:, 1:] = -a[:, :0:-1]


def test_threads_and_contexts(ctx):
    g = workloads.rng(77)
    other = enchip.Context(0)
    errors = []

    def run(c, seed):
        try:
            r = workloads.rng(seed)
            for i in range(6):
                M = int(r.integers(700, 4000))
                a = r.integers(-127, 128, size=(M, 1501)).astype(np.float32)
                a[:, 0] = 127
                codes, _ = c.quant_rows(a)
                if not np.array_equal(codes, a.astype(np.int8)):
                    errors.append((seed, i, M))
        except Exception as e:  # noqa: BLE001 -- reported by the main thread
            errors.append((seed, repr(e)))

    threads = [threading.Thread(target=run, args=(c, int(s))) for c, s in
               zip([ctx, ctx, other, other], g.integers(0, 1 << 30, size=4))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    other.close()
    assert not errors, errors


def host_calls(ctx):
    # results of 600 KiB and of 3 MiB, inputs of 6 MiB, top-k hits
    g = workloads.rng(55)
    out = []
    for M, K, N in ((200, 64, 768), (1536, 1024, 512)):
        w = ctx.register_weight(*workloads.int8_weights(g, N, K))
        out.append(ctx.linear(w, workloads.activations(g, M, K)))
    out += list(ctx.quant_rows(workloads.activations(g, 1100, 512)))
    out.append(ctx.matmul_bt_f32(workloads.activations(g, 300, 96), workloads.activations(g, 700, 96)))
    out += list(ctx.ann_topk(w, workloads.activations(g, 5, 1024), 7))
    return out


SHIM = "int hipHostMalloc(void **p, unsigned long n, unsigned f) { if (p) *p = 0; ++calls; return 2; }"


def test_without_pinned_memory_the_copies_are_pageable(ctx, tmp_path):
    # A process whose pinned allocations fail (a hipHostMalloc that answers out of memory stands
    # before the runtime's) gets the results of one that has them.
    (tmp_path / "shim.c").write_text("int calls;\n" + SHIM)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(tmp_path / "shim.so"), str(tmp_path / "shim.c")], check=True)
    child = f"""
import ctypes
shim = ctypes.CDLL({str(tmp_path / 'shim.so')!r}, mode=ctypes.RTLD_GLOBAL)
import numpy as np
from aikit_amd import enchip, workloads
{inspect.getsource(host_calls)}
with enchip.Context(0) as c:
    out = host_calls(c)
assert ctypes.c_int.in_dll(shim, "calls").value > 0, "the library's allocations did not fail"
np.savez({str(tmp_path / 'out.npz')!r}, *out)
"""
    print("[case] host copies without pinned memory", flush=True)
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", child], cwd=root, timeout=100, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    with np.load(tmp_path / "out.npz") as got:
        for i, want in enumerate(host_calls(ctx)):
            assert np.array_equal(got[f"arr_{i}"].view(np.uint8), np.ascontiguousarray(want).view(np.uint8)), i
