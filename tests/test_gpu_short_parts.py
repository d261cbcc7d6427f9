"""The resident kernel's parts of fewer than four slices: K of one to three slices, and of 5, 6 and 9, which is cut evenly (one block, whole slices,
a block more), with one wave and with two to a pair of tiles and with two pairs to a wave, against the oracle's product in f64."""
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


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,n", [(16, 257), (33, 600)])
@pytest.mark.parametrize("k", [32, 256, 288, 512, 544, 768, 1024, 1056, 1280, 1312, 1536, 2080, 2304])
def test_short_parts(ctx, orc, fmt, m, n, k):
    """Bound: f32 activations enter as two fp16 that are cut, not rounded, after 11 bits each: each cut leaves out less than 2^-10 of what it cuts, so
    2^-20 of an activation at most (fp16 activations: nothing); f32 sums whose roundings of 2^-24 grow like a random walk; both on quants whose sums
    are up to five times the product's."""
    w = synth.normal(k + n, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(m + k, m * k).reshape(m, k).copy(), synth.normal(7, m * n).reshape(m, n)
    x[0], x[1], x[2, : k // 2] = 0, x[1] * 2.0 ** -10, x[2, : k // 2] * 2.0 ** -6
    dq = orc.dequantize(fmt, orc.quantize(fmt, w), k, n)
    wt, db, c = ctx.weight(fmt, w), ctx.upload(d), ctx.buffer(m * n * 4)
    # (forced: one wave to a pair; the library's choice: two or four where the launch leaves CUs idle; fp16: row groups of 16 only up to 16 rows)
    for dtype, route in ((np.float32, capi.ROUTE_TILE_MFMA), (np.float32, capi.ROUTE_AUTO), (np.float16, capi.ROUTE_TILE_MFMA)):
        xa = x.astype(dtype)
        exact = orc.matmul_f64(xa.astype(np.float32), dq)
        cut = 0.0 if dtype == np.float16 else 2.0 ** -20
        bound = 5 * 0.02 * np.sqrt(n) * (cut + 2.0 ** -23 + 2.0 ** -24 * np.sqrt(k)) * np.linalg.norm(xa.astype(np.float64), axis=1) + 1e-30
        a = ctx.upload(xa)
        ctx.set_route(route)
        try:
            got = []
            for res in (None, None, db):
                (ctx.matmul_q_f16a if dtype == np.float16 else ctx.matmul_q)(a, wt, c, m, res)
                got.append(c.download(np.float32, m * n).reshape(m, n))
        finally:
            ctx.set_route(capi.ROUTE_AUTO)
            a.free()
        assert (np.linalg.norm(got[0] - exact, axis=1) <= bound).all(), (dtype, route)
        assert (bits(got[0]) == bits(got[1])).all()
        np.testing.assert_array_equal(got[2], got[0] + d)
    for h in (wt, db, c):
        h.free()


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n,f16", [(400, 256, 2700, False), (401, 288, 2700, False), (400, 544, 2690, False), (389, 1056, 2182, False), (385, 1536, 2177, False),
                                       (390, 1024, 2700, False), (5, 288, 66000, True)])
def test_two_pairs_of_tiles_per_wave(ctx, orc, fmt, m, k, n, f16):
    """The bound above."""
    if not f16:
        p = capi.matmul_plan(fmt, m, k, n)
        assert p.route == capi.ROUTE_TILE_MFMA and p.waves_n == 32 and p.quads_per_wave == 0
    w = synth.normal(k + n, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(m + k, m * k).reshape(m, k).copy(), synth.normal(7, m * n).reshape(m, n)
    x[0], x[1] = 0, x[1] * 2.0 ** -10
    x = x.astype(np.float16) if f16 else x
    exact = orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    wt, a, c, db = ctx.weight(fmt, w), ctx.upload(x), ctx.buffer(m * n * 4), ctx.upload(d)
    ctx.set_route(capi.ROUTE_TILE_MFMA)
    try:
        got = []
        for res in (None, None, db):
            (ctx.matmul_q_f16a if f16 else ctx.matmul_q)(a, wt, c, m, res)
            got.append(c.download(np.float32, m * n).reshape(m, n))
    finally:
        ctx.set_route(capi.ROUTE_AUTO)
        for h in (wt, a, c, db):
            h.free()
    cut = 0.0 if f16 else 2.0 ** -20
    bound = 5 * 0.02 * np.sqrt(n) * (cut + 2.0 ** -23 + 2.0 ** -24 * np.sqrt(k)) * np.linalg.norm(x.astype(np.float64), axis=1) + 1e-30
    assert (np.linalg.norm(got[0] - exact, axis=1) <= bound).all()
    assert (bits(got[0]) == bits(got[1])).all()
    np.testing.assert_array_equal(got[2], got[0] + d)
