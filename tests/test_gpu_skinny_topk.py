"""GPU tests of the candidate kernel behind the fused top-k at its edges: against the oracle's
scores and the reference's selection, exactly (ids, order and score bits)."""
import numpy as np
import oracle
import pytest

from aikit_amd import workloads

pytestmark = pytest.mark.gpu


# rows: one, two, four and eight row blocks a launch, ragged; a launch of one row after 256.
# K: 4, 8, 12 and 16 K steps. N % 64 in {0, 4, 36}: the last pair of channel groups ragged.
# k = 1, and 64 (a workgroup's slots for a row overflow into the global lists).
@pytest.mark.parametrize("M,N,K,k", [(33, 131072, 128, 10), (128, 131076, 256, 1), (129, 131108, 384, 10),
                                     (256, 131076, 512, 10), (257, 150004, 100, 10), (200, 262144, 384, 64),
                                     (8, 131108, 512, 64)])
@pytest.mark.parametrize("odd", [False, True])
def test_candidates_match_oracle(ctx, M, N, K, k, odd):
    # odd: query rows of zeros and of scales outside the fast comparison's range (codes of
    # subnormal and of very large values), index scales that are negative, zero, infinite, NaN,
    # subnormal, and sign-flipped copies of index rows (ties of both signs).
    g = workloads.rng(7100 + M + N + K + k)
    q = workloads.activations(g, M, K)
    codes = g.integers(-127, 128, size=(N, K), dtype=np.int8)
    scales = g.uniform(1e-3, 1e-2, size=N).astype(np.float32)
    if odd:
        q[0] = 0
        q[M // 2] *= np.float32(2.0 ** -110)
        q[M - 1] *= np.float32(2.0 ** 60)
        scales[g.random(N) < 0.2] *= -1
        for v in (0.0, np.inf, -np.inf, np.nan, 1e-42):
            scales[g.random(N) < 2e-5] = v
        codes[N // 2:N // 2 + 4096] = -codes[:4096]
        scales[N // 2:N // 2 + 4096] = -scales[:4096]
    print(f"[case] skinny candidates M={M} N={N} K={K} k={k} odd={odd}", flush=True)
    w = ctx.register_weight(codes, scales)
    try:
        f0, _ = ctx.ann_topk_stats()
        hi, hs = ctx.ann_topk(w, q, k)
        f1, _ = ctx.ann_topk_stats()
    finally:
        ctx.release_weight(w)
    assert f1 == f0 + 1, "route"
    with np.errstate(all="ignore"):
        scores = oracle.w8a8_linear(q, codes, scales, None, 0, M, K, N)
    for r in range(M):
        idx, sc = oracle.top_hits(scores[r], k)
        assert hi[r, :idx.size].tolist() == idx.tolist(), f"row {r}: indices differ"
        assert np.array_equal(hs[r, :idx.size].view(np.uint32), sc.view(np.uint32)), f"row {r}: scores differ"
        assert (hi[r, idx.size:] == -1).all() and np.isnan(hs[r, idx.size:]).all(), f"row {r}: padding"


@pytest.mark.parametrize("k,live", [(10, 10), (10, 9), (64, 1024)])
def test_bounds_of_few_live_groups(ctx, k, live):
    # NaN index scales leave `live` of the sample's 1024 column groups a score: the k-th largest
    # group maximum, or no bound where fewer than k have one (every score is listed, the lists
    # overflow and the two-pass route answers). Equal codes, so ties go by index.
    M, N, K = 40, 131072, 128
    g = workloads.rng(7900 + k + live)
    q = np.abs(workloads.activations(g, M, K)) + np.float32(0.01)
    codes = np.ones((N, K), np.int8)
    scales = np.full(N, 1e-3, np.float32)
    sample = np.full((1024, 32), np.nan, np.float32)
    sample[g.permutation(1024)[:live], g.integers(0, 32)] = 2e-3
    scales[:32768] = sample.reshape(-1)
    print(f"[case] skinny bounds k={k} live={live}", flush=True)
    w = ctx.register_weight(codes, scales)
    try:
        _, b0 = ctx.ann_topk_stats()
        hi, hs = ctx.ann_topk(w, q, k)
        _, b1 = ctx.ann_topk_stats()
    finally:
        ctx.release_weight(w)
    assert b1 - b0 == (1 if live < k else 0), "route"
    scores = oracle.w8a8_linear(q, codes, scales, None, 0, M, K, N)
    for r in range(M):
        idx, sc = oracle.top_hits(scores[r], k)
        assert hi[r].tolist() == idx.tolist(), f"row {r}: indices differ"
        assert np.array_equal(hs[r].view(np.uint32), sc.view(np.uint32)), f"row {r}: scores differ"


@pytest.mark.parametrize("M,N,K,k,doc", [(8, 1 << 20, 128, 32, 32), (40, 1 << 20, 128, 32, 16), (130, 1 << 19, 128, 64, 32)])
def test_rows_stored_by_document_stay_on_the_fused_route(ctx, M, N, K, k, doc):
    # `doc` consecutive rows score alike (correlation 0.9), as the passages of a document stored in
    # order do: the bounds are as tight as over any order, so the lists hold and the fused route
    # answers. Taken over 32 adjacent columns the group maxima would let too many through.
    g = workloads.rng(8100 + M + doc)
    x = np.repeat(g.standard_normal((N // doc, K), dtype=np.float32), doc, axis=0) * np.float32(0.9**0.5)
    x += g.standard_normal((N, K), dtype=np.float32) * np.float32(0.1**0.5)
    codes = np.clip(np.rint(x * 30), -127, 127).astype(np.int8)
    del x
    scales = np.full(N, 1e-3, np.float32)
    q = g.standard_normal((M, K)).astype(np.float32)
    print(f"[case] ann by document M={M} N={N} K={K} k={k} doc={doc}", flush=True)
    w = ctx.register_weight(codes, scales)
    try:
        f0, b0 = ctx.ann_topk_stats()
        hi, hs = ctx.ann_topk(w, q, k)
        f1, b1 = ctx.ann_topk_stats()
    finally:
        ctx.release_weight(w)
    scores = oracle.w8a8_linear(q, codes, scales, None, 0, M, K, N)
    sample, cap = scores[:, :32768], 4096 if k <= 32 else 8192

    def longest(groups):
        kth = -np.partition(-groups, k - 1, axis=1)[:, k - 1]
        return int((scores >= kth[:, None]).sum(axis=1).max())

    assert longest(sample) <= cap < longest(sample.reshape(M, 1024, 32).max(axis=2)), "the case"
    assert (f1 - f0, b1 - b0) == (1, 0), "route"
    for r in range(M):
        idx, sc = oracle.top_hits(scores[r], k)
        assert hi[r].tolist() == idx.tolist(), f"row {r}: indices differ"
        assert np.array_equal(hs[r].view(np.uint32), sc.view(np.uint32)), f"row {r}: scores differ"
