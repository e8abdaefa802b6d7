"""GPU tests of the f32 MatmulBT's split products (three bf16 parts per operand, six products):
every tile form at its edges against float64 with the bound its roundings give, operands the
split cannot hold, and one result per problem whatever the batch and layout."""
import numpy as np
import pytest

from aikit_amd import enchip, workloads

pytestmark = pytest.mark.gpu

# (M, K, N): the K split in 32 x 32, 64 x 32 and 64 x 64 tiles; 64 x 64, 64 x 128, 128 x 64
# and 128 x 128 tiles; with remainders in every dimension, K below and past a chunk, and
# K or N not a multiple of 4 (values loaded one by one)
SHAPES = [(33, 300, 132, "k32"), (500, 257, 1000, "k64x32"), (1, 1024, 4097, "k"), (70, 40, 100, "64"), (65, 33, 65, "64"),
          (500, 200, 2050, "64x128"), (3000, 100, 60, "128x64"), (1200, 96, 1500, "128x64"), (2100, 52, 2052, "128"),
          (1999, 31, 2301, "128"), (2, 5, 3, "64")]


def bound(a, b, K):
    """|C - exact| <= (adds + 2) 2^-24 sum |a b|: 6 rounded adds of the running sum per 16-deep
    step, the K split's 3 and the products left out (together under 2^-24 |a b|)."""
    return (6 * -(-K // 16) + 3 + 2) * 2.0**-24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T)


@pytest.mark.parametrize("M,K,N,form", SHAPES)
@pytest.mark.parametrize("layout", [enchip.B_NK, enchip.B_KN])
def test_split_products_within_their_rounding_bound(ctx, M, K, N, form, layout):
    import torch

    g = workloads.rng(5000 + M + K + N)
    a = g.standard_normal((M, K)).astype(np.float32)
    b = g.standard_normal((N, K)).astype(np.float32)
    a *= np.exp2(g.integers(-8, 9, size=(M, K))).astype(np.float32)  # a spread of magnitudes
    print(f"[case] f32 split M={M} K={K} N={N} layout={layout} ({form})", flush=True)
    da = torch.from_numpy(a).cuda()
    db = torch.from_numpy(np.ascontiguousarray(b if layout == enchip.B_NK else b.T)).cuda()
    dc = torch.full((M, N), 7.0, device="cuda")
    torch.cuda.synchronize()
    ctx.matmul_bt_f32_dev(da.data_ptr(), K, db.data_ptr(), K if layout == enchip.B_NK else N, layout, dc.data_ptr(), N,
                          M, K, N)
    torch.cuda.synchronize()
    ref = a.astype(np.float64) @ b.astype(np.float64).T
    assert np.all(np.abs(dc.cpu().numpy() - ref) <= bound(a, b, K))


@pytest.mark.parametrize("M,K,N", [(100, 300, 200), (80, 64, 70), (2100, 64, 2052)])
def test_infinities_nans_and_the_largest_floats(ctx, M, K, N):
    # What f32 arithmetic gives: an infinity times a nonzero value is an infinity, times zero
    # NaN; a float that rounds to infinity in bf16 stays finite; the other rows are untouched.
    g = workloads.rng(77 + M)
    a = g.standard_normal((M, K)).astype(np.float32)
    b = np.abs(g.standard_normal((N, K))).astype(np.float32) + np.float32(0.5)
    a[3, 5] = np.inf
    a[7, K - 1] = -np.inf
    a[11, 2] = np.nan
    a[M - 1] = 0
    a[M - 1, 1] = np.float32(3.4028235e38)  # the largest float, times 0.5 .. : finite or inf as f32 has it
    b[4, 5] = 0  # inf * 0
    b[N - 1, 1] = np.float32(0.25)
    with np.errstate(all="ignore"):
        want = (a.astype(np.float64)[:, None, :] * b.astype(np.float64)[None, :, :]).sum(-1) if M < 1000 else None
        got = ctx.matmul_bt_f32(a, b)
        assert np.all(np.isposinf(np.delete(got[3], 4))) and np.isnan(got[3, 4])
        assert np.all(np.isneginf(got[7])) and np.all(np.isnan(got[11]))
        big = np.float32(3.4028235e38) * b[:, 1]  # one product: its f32 rounding, infinities included
        assert np.array_equal(got[M - 1], big)
        rows = np.setdiff1d(np.arange(M), [3, 7, 11, M - 1])
        if want is not None:
            # blocks that hold a special value run on the f32 MFMA: at most one rounded add per product
            f32 = (K + 2) * 2.0**-24 * (np.abs(a[rows]).astype(np.float64) @ np.abs(b).astype(np.float64).T)
            assert np.all(np.abs(got[rows] - want[rows]) <= f32)
        assert np.isfinite(got[rows]).all()


def test_a_batch_gives_each_problem_its_own_bits(ctx):
    # 40 problems of one shape in a launch (larger tiles than one alone would get) and one by one
    import torch

    g = workloads.rng(9)
    for M, K, N in ((96, 512, 160), (130, 300, 64), (64, 64, 128)):
        a = torch.from_numpy(g.standard_normal((40, M, K)).astype(np.float32)).cuda()
        b = torch.from_numpy(g.standard_normal((40, N, K)).astype(np.float32)).cuda()
        c1, c2 = torch.empty((40, M, N), device="cuda"), torch.empty((40, M, N), device="cuda")
        torch.cuda.synchronize()
        print(f"[case] batch of 40 M={M} K={K} N={N}", flush=True)
        ctx.matmul_bt_f32_dev(a.data_ptr(), K, b.data_ptr(), K, enchip.B_NK, c1.data_ptr(), N, M, K, N,
                              inner=(40, M * K, N * K, M * N))
        for i in range(40):
            ctx.matmul_bt_f32_dev(a[i].data_ptr(), K, b[i].data_ptr(), K, enchip.B_NK, c2[i].data_ptr(), N, M, K, N)
        torch.cuda.synchronize()
        assert torch.equal(c1.view(torch.int32), c2.view(torch.int32))


def product(ctx, a, b, layout):
    """a[M, K] . b[N, K]^T from device buffers, B in either layout."""
    import torch

    (M, K), N = a.shape, b.shape[0]
    da = torch.from_numpy(a).cuda()
    db = torch.from_numpy(np.ascontiguousarray(b if layout == enchip.B_NK else b.T)).cuda()
    dc = torch.full((M, N), 7.0, device="cuda")
    torch.cuda.synchronize()
    ctx.matmul_bt_f32_dev(da.data_ptr(), K, db.data_ptr(), K if layout == enchip.B_NK else N, layout, dc.data_ptr(), N,
                          M, K, N)
    torch.cuda.synchronize()
    return dc.cpu().numpy()


@pytest.mark.parametrize("M,K,N", [(130, 300, 200), (40, 512, 160), (300, 64, 300), (65, 40, 100), (1200, 96, 1500)])
@pytest.mark.parametrize("bad", [np.inf, np.nan, 3.4e38])
def test_outputs_beside_a_special_value_keep_their_bits(ctx, M, K, N, bad):
    # one row of A and one of B hold a value the split cannot: every other output has the bits of
    # the product without them, in one problem and in a batch of 24 (other tile sizes)
    import torch

    g = workloads.rng(6500 + M)
    a, b = g.standard_normal((M, K)).astype(np.float32), g.standard_normal((N, K)).astype(np.float32)
    print(f"[case] f32 beside {bad} M={M} K={K} N={N}", flush=True)
    clean = product(ctx, a, b, enchip.B_NK)
    i, j = M // 2, N // 3
    a[i, K // 2], b[j, 1] = bad, bad
    with np.errstate(all="ignore"):
        one = product(ctx, a, b, enchip.B_NK)
    keep = np.ones((M, N), bool)
    keep[i], keep[:, j] = False, False
    assert np.array_equal(one.view(np.int32)[keep], clean.view(np.int32)[keep])
    da, db = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    dc = torch.empty((24, M, N), device="cuda")
    torch.cuda.synchronize()
    ctx.matmul_bt_f32_dev(da.data_ptr(), K, db.data_ptr(), K, enchip.B_NK, dc.data_ptr(), N, M, K, N,
                          inner=(24, 0, 0, M * N))
    torch.cuda.synchronize()
    assert np.array_equal(dc.cpu().numpy().view(np.int32), np.broadcast_to(one.view(np.int32), (24, M, N)))


@pytest.mark.parametrize("N", [256, 1031])
@pytest.mark.parametrize("layout", [enchip.B_NK, enchip.B_KN])
def test_partial_sums_that_overflow_together(ctx, N, layout):
    # K split over wavefronts: in 32-deep chunks 0, 2 and 5 (wavefronts 0, 2 and 1) 2e38, -2e38 and
    # 2e38. Adding the wavefronts' sums in their order overflows; f32 adds in k order do not.
    a = np.zeros((33, 1024), np.float32)
    a[::2, 0], a[::2, 64], a[::2, 160] = 2e38, -2e38, 2e38
    a[1::2] = np.float32(0.25)
    b = np.ones((N, 1024), np.float32)
    print(f"[case] f32 partial sums N={N} layout={layout}", flush=True)
    got = product(ctx, a, b, layout)
    assert (got[::2] == np.float32(2e38)).all() and (got[1::2] == 256).all()


# the K split in each tile size, then the tile forms; K and N multiples of 4 or not
@pytest.mark.parametrize("M,K,N", [(33, 300, 132), (500, 257, 1000), (130, 1024, 1031), (70, 40, 100), (500, 200, 2050),
                                   (1200, 96, 1500), (1999, 31, 2301)])
@pytest.mark.parametrize("layout", [enchip.B_NK, enchip.B_KN])
@pytest.mark.parametrize("ea,eb,where", [(-112, 110, "all"), (-120, 118, "all"), (-127, 120, "all"), (-140, 124, "few"),
                                         (118, -120, "all"), (120, -126, "few")])
def test_small_operands_keep_f32_precision(ctx, M, K, N, layout, ea, eb, where):
    # Operands near 2^ea and 2^eb, the small ones (f32 subnormals among them) too small for three
    # bf16 parts: everywhere, or a few of them among zeros and values of ordinary size. One
    # rounded add per product, and a product's rounding: (K + 2) 2^-24 sum |a b|, and 2^-149 a
    # product where it is subnormal.
    g = workloads.rng(6100 + M + ea)
    a = (1 + g.random((M, K))).astype(np.float32) * g.choice(np.float32([-1, 1]), size=(M, K))
    b = (1 + g.random((N, K))).astype(np.float32)
    small, big, es, eg = (a, b, ea, eb) if ea < eb else (b, a, eb, ea)
    if where == "all":
        small[:] = np.ldexp(small, es)
        big[:] = np.ldexp(big, eg)
    else:
        few = g.random(small.shape) < 2.0 / K
        few[: small.shape[0] // 2] = False
        small[:] = np.where(few, np.ldexp(small, es), np.where(g.random(small.shape) < 0.5, 0, small))
        big[:, :] = np.where(g.random(big.shape) < 0.5, np.ldexp(big, eg - 20), np.ldexp(big, -100))
    print(f"[case] f32 small operands M={M} K={K} N={N} layout={layout} 2^{ea} 2^{eb} {where}", flush=True)
    got = product(ctx, a, b, layout)
    ref = a.astype(np.float64) @ b.astype(np.float64).T
    lim = (K + 2) * 2.0**-24 * (np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T) + K * 2.0**-149
    assert np.all(np.abs(got - ref) <= lim)


@pytest.mark.parametrize("M,K,N", [(96, 512, 160), (300, 64, 300), (40, 24, 2500)])
def test_small_operands_beside_others_in_any_tile(ctx, M, K, N):
    # 24 problems in a launch and one by one (other tile sizes): small operands in a few rows of A
    # and of B, zero rows beside them, one value above 2^24: the same bits for every output.
    import torch

    g = workloads.rng(6900 + M)
    a = g.standard_normal((24, M, K)).astype(np.float32)
    b = g.standard_normal((24, N, K)).astype(np.float32)
    for p in range(24):
        a[p, g.integers(0, M, 3)] = 0
        a[p, g.integers(0, M, 3), g.integers(0, K, 3)] = np.float32(2.0**-125 * 1.7)
        a[p, g.integers(0, M)] *= np.float32(2.0**-115)
        b[p, g.integers(0, N), g.integers(0, K)] = np.float32(2.0**100 if p % 2 else -(2.0**-149))
    da, db = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    c1, c2 = torch.empty((24, M, N), device="cuda"), torch.empty((24, M, N), device="cuda")
    torch.cuda.synchronize()
    print(f"[case] f32 small operands, batch of 24 M={M} K={K} N={N}", flush=True)
    ctx.matmul_bt_f32_dev(da.data_ptr(), K, db.data_ptr(), K, enchip.B_NK, c1.data_ptr(), N, M, K, N,
                          inner=(24, M * K, N * K, M * N))
    for i in range(24):
        ctx.matmul_bt_f32_dev(da[i].data_ptr(), K, db[i].data_ptr(), K, enchip.B_NK, c2[i].data_ptr(), N, M, K, N)
    torch.cuda.synchronize()
    assert torch.equal(c1.view(torch.int32), c2.view(torch.int32))
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    ref = np.matmul(a64, b64.transpose(0, 2, 1))
    lim = (6 * -(-K // 16) + 6 + K) * 2.0**-24 * np.matmul(np.abs(a64), np.abs(b64).transpose(0, 2, 1)) + K * 2.0**-149
    assert np.all(np.abs(c1.cpu().numpy() - ref) <= lim)
