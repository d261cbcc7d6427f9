"""The resident kernel's launches whose waves split K (small calls of more than four rows): at the edges of slices, K parts, row
groups of 8 and 16, column groups and formats, against the oracle's product in f64 and against the same kernel
without the split (the forced route)."""
import numpy as np
import pytest

from helpers import Q4, Q8, bits
from meganeura_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = capi.Context(0)
    yield c
    c.close()


def rows_of(m, k, seed):
    """Ordinary rows, and among them zeros, tiny and large ones and one whose slices are far apart."""
    x = synth.normal(seed, m * k).reshape(m, k).copy()
    x[0] = 0
    x[1] *= 1e-12
    x[m - 1] *= 1e9
    x[m - 2, : k // 2] *= 1e-4
    return x


def run(ctx, x, wt, d=None, ops=(), route=capi.ROUTE_AUTO, static=False):
    m, n = len(x), wt.cols
    a, c = ctx.upload(x), ctx.buffer(m * n * 4)
    db = None if d is None else ctx.upload(d)
    ctx.set_route(route)
    try:
        if x.dtype == np.float16:
            ctx.matmul_q_f16a(a, wt, c, m, db)
        elif static:
            ctx.matmul_q_static(a, wt, c, m, db)
        else:
            ctx.matmul_q_epilogue(a, wt, c, m, list(ops), db)
        return c.download(np.float32, m * n).reshape(m, n)
    finally:
        ctx.set_route(capi.ROUTE_AUTO)
        for b in (a, c, db):
            if b is not None:
                b.free()


# (m, k, n, waves that share a pair of tiles, K parts): by K, one slice more and one block less
SHAPES = [(5, 288, 64, 2, 1), (8, 512, 129, 2, 1), (9, 544, 65, 4, 1), (16, 768, 1, 4, 1), (17, 1024, 63, 4, 1), (24, 1056, 200, 4, 2),
          (33, 992, 517, 4, 1), (31, 3104, 96, 4, 4), (6, 8224, 40, 4, 9), (77, 576, 1000, 4, 1), (16, 320, 1856, 2, 1), (300, 544, 33, 4, 1)]


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n,ks,parts", SHAPES)
def test_against_the_oracle_and_without_the_split(ctx, orc, fmt, m, k, n, ks, parts):
    """Both add the same exact products of 22-bit activations (relative to a slice's largest) in f32, in another order of the slices:
    roundings of 2^-24 each on sums that grow like a random walk, 2^-24 sqrt(K) of their size, and the 2^-22 of the activations against
    f64.  The products enter with nibbles of 0 .. 15 and bytes of 0 .. 255 (the minima and the bias come after): for normal weights those sums
    are up to five times the row's size, five times the above."""
    p = capi.matmul_plan(fmt, m, k, n, auto=True)
    assert (p.route, p.k_splits, p.k_parts) == (capi.ROUTE_TILE_MFMA, ks, parts)
    w = synth.normal(2 * k + n, k * n, 0.02).reshape(k, n)
    x, d = rows_of(m, k, m + k), synth.normal(7, m * n).reshape(m, n)
    wt = ctx.weight(fmt, w)
    exact = orc.matmul_f64(x, orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    got = [run(ctx, x, wt) for _ in range(3)]
    assert (bits(got[0]) == bits(got[1])).all() and (bits(got[0]) == bits(got[2])).all()
    bound = 5 * (2.0 ** -22 + 2.0 ** -24 * np.sqrt(k))
    size = 0.02 * np.linalg.norm(x.astype(np.float64), axis=1) * np.sqrt(n) + 1e-30
    behind = run(ctx, x, wt, route=capi.ROUTE_TILE_MFMA)
    for want in (exact, behind.astype(np.float64)):
        assert (np.linalg.norm(got[0] - want, axis=1) <= bound * size).all()
    # the residual and the unary operations come last
    with_d = run(ctx, x, wt, d)
    np.testing.assert_array_equal(with_d, got[0] + d)
    np.testing.assert_array_equal(run(ctx, x, wt, d, [capi.UNARY_NEG, capi.UNARY_RELU]), np.maximum(-with_d, 0))
    np.testing.assert_array_equal(run(ctx, x, wt, d, static=True), with_d)
    wt.free()


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n", [(5, 544, 64), (9, 768, 65), (18, 2080, 201), (40, 992, 300), (107, 4000, 256)])
def test_fp16_activations(ctx, orc, fmt, m, k, n):
    """fp16 activations enter exactly: f32 sums of K products and block means carried with 22 bits, on the same sums as above."""
    p = capi.matmul_plan(fmt, m, k, n, True, auto=True)
    assert p.route == capi.ROUTE_TILE_MFMA and p.k_splits == 4
    w = synth.normal(k + n, k * n, 0.02).reshape(k, n)
    x = synth.normal(m, m * k).reshape(m, k).astype(np.float16)
    x[0], x[1] = 0, x[1] * np.float16(2.0 ** -10)
    wt = ctx.weight(fmt, w)
    exact = orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    size = 0.02 * np.linalg.norm(x.astype(np.float64), axis=1) * np.sqrt(n) + 1e-30
    assert (np.linalg.norm(run(ctx, x, wt) - exact, axis=1) <= 5 * (2.0 ** -22 + 2.0 ** -24 * np.sqrt(k)) * size).all()
    wt.free()


def check(ctx, orc, fmt, x, n):
    """Results, repeats, residual and rows that are not finite, against f64 and against the kernel without the split; bounds as above."""
    m, k = x.shape
    w, d = synth.normal(2 * k + n, k * n, 0.02).reshape(k, n), synth.normal(7, m * n).reshape(m, n)
    wt = ctx.weight(fmt, w)
    exact = orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    size = 0.02 * np.linalg.norm(x.astype(np.float64), axis=1) * np.sqrt(n) + 1e-30
    got = run(ctx, x, wt)
    for want in (exact, run(ctx, x, wt, route=capi.ROUTE_TILE_MFMA).astype(np.float64)):
        assert (np.linalg.norm(got - want, axis=1) <= 5 * (2.0 ** -22 + 2.0 ** -24 * np.sqrt(k)) * size).all()
    for _ in range(2):
        assert (bits(run(ctx, x, wt)) == bits(got)).all()
    np.testing.assert_array_equal(run(ctx, x, wt, d), got + d)
    y = x.copy()
    y[1, 3], y[2, k - 1], y[m - 1, 300] = np.nan, np.inf, -np.inf
    wrong, bad = run(ctx, y, wt), [1, 2, m - 1]
    good = [r for r in range(m) if r not in bad]
    assert not np.isfinite(wrong[bad]).any()
    np.testing.assert_array_equal(wrong[good], got[good])
    wt.free()


@pytest.mark.parametrize("fmt,m,k,n,f16,parts", [
    (Q4, 101, 704, 2409, False, 1), (Q4, 200, 928, 1418, False, 1), (Q8, 101, 704, 2561, False, 1), (Q8, 200, 992, 1457, False, 1),
    (Q8, 76, 1312, 1796, False, 2), (Q8, 200, 1056, 588, False, 2), (Q8, 101, 2080, 1029, False, 3), (Q8, 76, 2528, 1098, False, 3),
    (Q4, 50, 576, 5580, True, 1), (Q4, 101, 1024, 2764, True, 1), (Q8, 200, 576, 1600, True, 1), (Q8, 200, 896, 1600, True, 1),
    (Q8, 101, 1184, 1293, True, 2), (Q8, 101, 1536, 1243, True, 2), (Q8, 101, 2240, 825, True, 3), (Q8, 101, 2336, 1184, True, 3)])
def test_two_waves_of_two_slices(ctx, orc, fmt, m, k, n, f16, parts):
    """Two waves to a pair of tiles, more than one slice each: parts of three (two and one) and four slices, the last of them two to four."""
    p = capi.matmul_plan(fmt, m, k, n, f16, auto=True)
    assert (p.route, p.k_splits, p.k_parts, p.steps) == (capi.ROUTE_TILE_MFMA, 2, parts, 2)
    x = rows_of(m, k, m + k) if not f16 else synth.normal(m, m * k).reshape(m, k).astype(np.float16)
    check(ctx, orc, fmt, x, n)


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n", [(5, 544, 64), (18, 2080, 201), (107, 4000, 256)])
def test_four_waves_with_fp16_activations(ctx, orc, fmt, m, k, n):
    p = capi.matmul_plan(fmt, m, k, n, True, auto=True)
    assert p.route == capi.ROUTE_TILE_MFMA and p.k_splits == 4
    check(ctx, orc, fmt, synth.normal(m, m * k).reshape(m, k).astype(np.float16), n)


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k", [(6, 544), (16, 1056), (20, 768)])
def test_values_that_are_not_finite_stay_in_their_rows(ctx, orc, fmt, m, k):
    n = 70
    w = synth.normal(k, k * n, 0.02).reshape(k, n)
    x = synth.normal(m, m * k).reshape(m, k).copy()
    clean = run(ctx, x, ctx.weight(fmt, w))
    x[1, 3], x[2, k - 1], x[m - 1, 300], x[4, 40] = np.nan, np.inf, -np.inf, 2.0 ** 101
    got = run(ctx, x, ctx.weight(fmt, w))
    bad = [1, 2, 4, m - 1]
    assert not np.isfinite(got[bad]).any()
    good = [r for r in range(m) if r not in bad]
    np.testing.assert_array_equal(got[good], clean[good])


def test_a_part_that_gives_up_is_reported(ctx, orc):
    m, k, n = 9, 2080, 128
    p = capi.matmul_plan(Q8, m, k, n, auto=True)
    assert p.k_splits == 4 and p.k_parts == 3
    w = synth.normal(1, k * n, 0.02).reshape(k, n)
    x = synth.normal(2, m * k).reshape(m, k)
    wt = ctx.weight(Q8, w)
    want = run(ctx, x, wt)
    a, c = ctx.upload(x), ctx.buffer(m * n * 4)
    try:
        ctx.set_spin_limit(0)
        ctx.matmul_q(a, wt, c, m)
        with pytest.raises(capi.MgnError) as e:
            ctx.sync()
        assert e.value.status == capi.ETIMEOUT
    finally:
        ctx.set_spin_limit(1 << 20)
    np.testing.assert_array_equal(run(ctx, x, wt), want)
    # a shared device: no parts that wait for each other
    ctx.set_shared_device(True)
    try:
        np.testing.assert_allclose(run(ctx, x, wt), want, rtol=2e-5, atol=2e-5)
    finally:
        ctx.set_shared_device(False)
    for h in (wt, a, c):
        h.free()
