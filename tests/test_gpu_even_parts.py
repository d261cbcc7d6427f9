"""K parts that go out evenly over the XCDs, where rounding a launch's groups up to a multiple of 8 would be another round of
workgroups, against the oracle's product in f64: the resident kernel one group before, at and behind the sizes at which its two grids part, the
blocked kernel with one tile, fewer than 8, and one more than a multiple of 8."""
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


# (m, k, n, fp16 activations, K parts, groups): a multiple of 8 in one round; 8 j + 1 and 8 j + 4 groups that only fit unrounded; the last that fit
SHAPES = [(320, 2080, 1024, False, 3, 80), (323, 2080, 1000, False, 3, 84), (5, 13344, 4097, False, 14, 17), (16, 10272, 5888, False, 11, 23),
          (17, 8224, 3580, False, 9, 28), (650, 2112, 900, True, 3, 84)]


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n,f16,parts,groups", SHAPES)
def test_parts_of_a_grid_that_is_not_rounded_up(ctx, orc, fmt, m, k, n, f16, parts, groups):
    """Normal data: products of activations with 22 bits (fp16 exactly), summed in f32 with roundings of 2^-24 that grow like a random walk,
    on sums up to five times the row's size (quants of 0 .. 15 and bytes of 0 .. 255; minima and bias come after)."""
    p = capi.matmul_plan(fmt, m, k, n, f16)
    if p.route != capi.ROUTE_TILE_MFMA:
        p = capi.matmul_plan(fmt, m, k, n)  # (fp16 on the forced route: the same groups, in row groups of 32)
    assert p.k_parts == parts and (f16 or p.grid[1] * p.grid[2] == groups)
    w = synth.normal(k + n, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(m + k, m * k).reshape(m, k), synth.normal(7, m * n).reshape(m, n)
    x = x.astype(np.float16) if f16 else x
    wt, a, c, db = ctx.weight(fmt, w), ctx.upload(x), ctx.buffer(m * n * 4), ctx.upload(d)
    exact = orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
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
    assert (bits(got[0]) == bits(got[1])).all()
    size = 0.02 * np.linalg.norm(x.astype(np.float64), axis=1) * np.sqrt(n)
    assert (np.linalg.norm(got[0] - exact, axis=1) <= 5 * (2.0 ** -22 + 2.0 ** -24 * np.sqrt(k)) * size).all()
    np.testing.assert_array_equal(got[2], got[0] + d)


# (m, k, n, fp16 activations)
BLOCKED = [(20, 4096, 100, False), (43, 8192, 1500, False), (96, 5120, 2306, False), (118, 6560, 1600, False), (200, 4160, 1300, True), (257, 2080, 2049, False)]


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n,f16", BLOCKED)
def test_blocked_tiles_of_all_parts_are_dealt_out_evenly(ctx, orc, fmt, m, k, n, f16):
    """The bound above, of which the blocked kernel's 23 bits need less."""
    p = capi.matmul_block_plan(fmt, m, k, n, f16)
    tiles = p.row_groups * p.col_groups
    assert p.k_parts > 1 and -(-tiles // 8) * p.k_parts > -(-tiles * p.k_parts // 8)
    w = synth.normal(k + n, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(m + k, m * k).reshape(m, k), synth.normal(7, m * n).reshape(m, n)
    x = x.astype(np.float16) if f16 else x
    wt, a, c, db = ctx.weight(fmt, w), ctx.upload(x), ctx.buffer(m * n * 4), ctx.upload(d)
    exact = orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    ctx.set_route(capi.ROUTE_BLOCK_MFMA)
    try:
        got = []
        for res in (None, db):
            c.upload(np.full(m * n, np.nan, np.float32))
            (ctx.matmul_q_f16a if f16 else ctx.matmul_q)(a, wt, c, m, res)
            got.append(c.download(np.float32, m * n).reshape(m, n))
    finally:
        ctx.set_route(capi.ROUTE_AUTO)
        for h in (wt, a, c, db):
            h.free()
    size = 0.02 * np.linalg.norm(x.astype(np.float64), axis=1) * np.sqrt(n)
    assert (np.linalg.norm(got[0] - exact, axis=1) <= 5 * (2.0 ** -22 + 2.0 ** -24 * np.sqrt(k)) * size).all()
    np.testing.assert_array_equal(got[1], got[0] + d)
