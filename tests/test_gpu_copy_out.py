"""GPU tests of the staged copy of results to host memory at the edges of its slices (512 KiB),
halves (2 MiB) and launches: every byte, from several threads and contexts."""
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
