"""Calls that the automatic route gives to the blocked kernel because of what the plan of the kernel behind it says (narrow results of long K, ragged
rounds), and calls with fp16 activations that it gives to the resident kernel in one round instead of the 32x32 one: every form of such a call on both
kernels, against the oracle's product in f64 and against each other."""
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


def run(ctx, x, wt, d=None, ops=(), route=capi.ROUTE_AUTO, static=False):
    m, n = len(x), wt.cols
    a, c = ctx.upload(x), ctx.upload(np.full(m * n, np.nan, np.float32))
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
        for h in (a, c, db):
            if h is not None:
                h.free()


@pytest.mark.parametrize("fmt,m,k,n,f16", [
    (Q4, 130, 4160, 992, False), (Q4, 51, 5056, 1088, False), (Q4, 399, 6656, 329, False), (Q8, 87, 1376, 11104, False), (Q8, 41, 5248, 1216, False),
    (Q8, 665, 6912, 575, False), (Q4, 546, 1056, 4423, True), (Q4, 267, 5440, 2279, True), (Q8, 949, 1120, 3090, True), (Q8, 1028, 5728, 911, True)])
def test_both_kernels_give_the_call_its_result(ctx, orc, fmt, m, k, n, f16):
    """Rows of ordinary, tiny, large and mixed magnitudes; bound: activations of 22 bits relative to a slice's largest, f32 sums whose roundings of
    2^-24 grow like a random walk, on sums up to five times the row's size, twice for the two kernels."""
    behind = capi.matmul_plan(fmt, m, k, n, f16).route
    assert capi.matmul_plan(fmt, m, k, n, f16, auto=True).route == capi.ROUTE_BLOCK_MFMA != behind
    w = synth.normal(2 * k + n, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(m + k, m * k).reshape(m, k).copy(), synth.normal(7, m * n).reshape(m, n)
    x[0] = 0
    if f16:
        x[1] *= 2.0 ** -10
        x = x.astype(np.float16)
    else:
        x[1] *= 1e-12
        x[m - 1] *= 1e9
        x[m - 2, : k // 2] *= 1e-4
    wt = ctx.weight(fmt, w)
    exact = orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    bound = 5 * (2.0 ** -22 + 2.0 ** -24 * np.sqrt(k)) * (0.02 * np.linalg.norm(x.astype(np.float64), axis=1) * np.sqrt(n) + 1e-30)
    got, other = run(ctx, x, wt), run(ctx, x, wt, route=behind)
    assert (np.linalg.norm(got - exact, axis=1) <= bound).all() and (np.linalg.norm(got.astype(np.float64) - other, axis=1) <= 2 * bound).all()
    assert (bits(run(ctx, x, wt)) == bits(got)).all()
    np.testing.assert_array_equal(run(ctx, x, wt, d), got + d)
    if not f16:
        np.testing.assert_array_equal(run(ctx, x, wt, d, [capi.UNARY_NEG, capi.UNARY_RELU]), np.maximum(-(got + d), 0))
        if capi.matmul_plan(fmt, m, k, n).workspace_bytes <= capi.STATIC_WORKSPACE_BYTES:
            np.testing.assert_array_equal(run(ctx, x, wt, d, static=True), got + d)
    # what is not finite stays in its rows
    x[1, 3], x[2, k - 1], x[m - 1, 300] = np.nan, np.inf, -np.inf
    bad = [1, 2, m - 1]
    for route in (capi.ROUTE_AUTO, behind):
        hit = run(ctx, x, wt, route=route)
        assert not np.isfinite(hit[bad]).any()
    good = [r for r in range(m) if r not in bad]
    np.testing.assert_array_equal(run(ctx, x, wt)[good], got[good])
    wt.free()


@pytest.mark.parametrize("fmt,m,k,n", [
    (Q4, 5, 8864, 1795), (Q4, 11, 7808, 4000), (Q4, 16, 1152, 21430), (Q4, 17, 10688, 2103), (Q4, 32, 3808, 2833), (Q8, 9, 4256, 5268), (Q8, 16, 1888, 17030),
    (Q8, 152, 3296, 394), (Q8, 308, 3072, 909), (Q8, 374, 1856, 1918)])
def test_fp16_activations_on_the_resident_kernel(ctx, orc, fmt, m, k, n):
    """fp16 activations enter exactly: f32 sums of K products and block means carried with 22 bits, on the same sums as above."""
    p = capi.matmul_plan(fmt, m, k, n, True, auto=True)
    assert p.route == capi.ROUTE_TILE_MFMA and p.k_splits == 1 and p.quads_per_wave == 0
    w = synth.normal(2 * k + n, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(m + k, m * k).reshape(m, k).astype(np.float16), synth.normal(7, m * n).reshape(m, n)
    x[0], x[1] = 0, x[1] * np.float16(2.0 ** -10)
    wt = ctx.weight(fmt, w)
    exact = orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    bound = 5 * (2.0 ** -22 + 2.0 ** -24 * np.sqrt(k)) * (0.02 * np.linalg.norm(x.astype(np.float64), axis=1) * np.sqrt(n) + 1e-30)
    got, other = run(ctx, x, wt), run(ctx, x, wt, route=capi.ROUTE_GEMM_MFMA)
    assert (np.linalg.norm(got - exact, axis=1) <= bound).all() and (np.linalg.norm(got.astype(np.float64) - other, axis=1) <= 2 * bound).all()
    assert (bits(run(ctx, x, wt)) == bits(got)).all()
    np.testing.assert_array_equal(run(ctx, x, wt, d), got + d)
    x[1, 3], x[2, k - 1], x[m - 1, 300] = np.nan, np.inf, -np.inf
    bad = [1, 2, m - 1]
    hit = run(ctx, x, wt)
    assert not np.isfinite(hit[bad]).any()
    good = [r for r in range(m) if r not in bad]
    np.testing.assert_array_equal(hit[good], got[good])
    # other work on the device: no parts that wait for each other
    ctx.set_shared_device(True)
    try:
        x[bad] = 0
        shared = run(ctx, x, wt)
        np.testing.assert_allclose(shared[good], got[good], rtol=0, atol=float(2 * bound.max()))
    finally:
        ctx.set_shared_device(False)
    wt.free()


@pytest.mark.parametrize("fmt,m,k,n", [(Q4, 547, 1216, 778), (Q4, 136, 1152, 4810), (Q8, 20, 1824, 479)])
def test_a_promise_that_does_not_hold_is_reported(ctx, fmt, m, k, n):
    """On a context that was promised activations in the fp16 range, these calls are the 32x32 and the blocked kernel's, which check them."""
    x = synth.normal(m + k, m * k).reshape(m, k).copy()
    wt = ctx.weight(fmt, synth.normal(2 * k + n, k * n, 0.02).reshape(k, n))
    ctx.set_activation_range(True)
    try:
        assert np.isfinite(run(ctx, x, wt)).all()
        x[m // 2, k - 1] = np.float32(70000.0)
        with pytest.raises(capi.MgnError) as e:
            run(ctx, x, wt)
        assert e.value.status == capi.ERANGE
        ctx.sync()  # reported once
    finally:
        ctx.set_activation_range(False)
    wt.free()


@pytest.mark.parametrize("fmt,m,k,n", [(Q8, 385, 1536, 2177), (Q8, 502, 224, 3873), (Q4, 403, 512, 3325), (Q4, 752, 32, 2513)])
def test_the_blocked_kernel_keeps_the_calls_that_it_answers_more_exactly(ctx, orc, fmt, m, k, n):
    """Calls on which the resident kernel would be the faster one, whose pairs of fp16 numbers are cut; the blocked kernel's are rounded to nearest.
    Measured 4 to 13 times the error; twice is asked for."""
    assert capi.matmul_plan(fmt, m, k, n, auto=True).route == capi.ROUTE_BLOCK_MFMA
    w, x = synth.normal(k + n, k * n, 0.02).reshape(k, n), synth.normal(m, m * k).reshape(m, k)
    wt = ctx.weight(fmt, w)
    exact = orc.matmul_f64(x, orc.dequantize(fmt, orc.quantize(fmt, w), k, n))
    error = [np.linalg.norm(run(ctx, x, wt, route=r) - exact) for r in (capi.ROUTE_AUTO, capi.ROUTE_TILE_MFMA)]
    assert 2 * error[0] <= error[1] <= 1e-5 * np.linalg.norm(exact)
    wt.free()
