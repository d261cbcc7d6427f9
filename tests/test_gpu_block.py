"""The blocked many-row kernel (MGN_ROUTE_BLOCK_MFMA) against the oracle, at the edges of what it is built
from: tiles of 32 rows and 64 columns, workgroups of 32 to 256 rows, blocks of 32 / stages of 64 or 128 / slices
of 256 elements of K, K parts; and rows whose magnitudes change along K."""
import os
import re

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


def run(ctx, x, wt, f16=False, d=None, ops=(), route=capi.ROUTE_BLOCK_MFMA):
    m, n = x.shape[0], wt.cols
    a, c = ctx.upload(x), ctx.buffer(m * n * 4)
    dd = ctx.upload(d) if d is not None else None
    ctx.set_route(route)
    try:
        if ops:
            ctx.matmul_q_epilogue(a, wt, c, m, list(ops), d=dd)
        else:
            (ctx.matmul_q_f16a if f16 else ctx.matmul_q)(a, wt, c, m, d=dd)
        return c.download(np.float32, m * n).reshape(m, n)
    finally:
        ctx.set_route(capi.ROUTE_AUTO)
        for b in (a, c) + ((dd,) if dd is not None else ()):
            b.free()


def assert_rows_close(got, want, x, k):
    """f32 accumulation of K products of 22-bit activations with exact weights: 2^-22 per product and 2^-24 per
    addition, both of the row's magnitude times the weights' (0.02, minima included 0.06) and, the errors
    being as good as independent, growing with sqrt(K); eight times that for the largest of many."""
    scale = np.abs(x).max(axis=1, keepdims=True).astype(np.float64)
    bound = 8 * (2.0**-22 + 2.0**-24) * 0.06 * np.sqrt(k) * scale
    assert np.isfinite(got).all()
    err = np.abs(got - want)
    assert (err <= bound + 2.0**-23 * np.abs(want)).all(), float((err / bound).max())


def mixed_rows(x):
    """Gives rows 3 to 8 slices of very different magnitudes: a large slice in front or at the end, small ones in the middle, and the
    three octaves around the one in which a row's scale is 1.  Returns the rows whose large part is the first 256 elements."""
    x[3, 256:] *= np.float32(2.0**-30)
    x[4, :-64] *= np.float32(2.0**-70)
    x[5, 700:900] *= np.float32(1e-20)
    for r, top in ((6, 9000.0), (7, 20000.0), (8, 40000.0)):
        x[r] *= np.float32(top / np.abs(x[r]).max())
        x[r, 256:] *= np.float32(2.0**-22)
    return [3, 6, 7, 8]


def tail_slice(k):
    return (k - 64) // 256 * 256


def assert_small_slices(got, want, x, dq, rows, first, last):
    """The small slices keep their own accuracy: in column `first`, whose weights are zero over the first 256 elements, and (row 4)
    column `last`, zero from the slice of the last 64 elements on."""
    k = x.shape[1]
    end = tail_slice(k)
    assert (dq[:256, first] == 0).all() and (dq[end:, last] == 0).all()
    assert_rows_close(got[rows, first][:, None], want[rows, first][:, None], x[rows, 256:], k)
    assert_rows_close(got[4:5, last][:, None], want[4:5, last][:, None], x[4:5, :end], k)


SHAPES = [(1, 32, 1), (31, 64, 63), (33, 96, 65), (32, 128, 64), (64, 160, 128), (65, 288, 257), (97, 992, 300), (129, 1056, 513),
          (200, 4064, 192), (257, 2048, 96), (77, 4096, 1000), (40, 16416, 70), (513, 320, 130)]


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("m,k,n", SHAPES)
def test_edges_of_tiles_stages_and_parts(ctx, orc, fmt, f16, m, k, n):
    w = synth.normal(2000 + fmt, k * n, 0.02).reshape(k, n)
    x = synth.normal(2001 + m, m * k).reshape(m, k)
    x = x.astype(np.float16) if f16 else x
    packed = orc.quantize(fmt, w)
    want = np.asarray(orc.matmul_f64(x.astype(np.float32), orc.dequantize(fmt, packed, k, n)), np.float64)
    wt = ctx.weight(fmt, w)
    got = run(ctx, x, wt, f16)
    assert_rows_close(got, want, x.astype(np.float32), k)
    assert np.array_equal(bits(run(ctx, x, wt, f16)), bits(got)), "not repeatable"
    wt.free()


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n", [(70, 2048, 4096), (50, 96, 70)])  # K in parts, K in one part
def test_residual_and_epilogue(ctx, orc, fmt, m, k, n):
    w = synth.normal(2010, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(2011, m * k).reshape(m, k), synth.normal(2012, m * n).reshape(m, n)
    wt = ctx.weight(fmt, w)
    want = orc.matmul_f32(x, orc.dequantize(fmt, orc.quantize(fmt, w), k, n), d).astype(np.float64)
    orc.assert_close(run(ctx, x, wt, d=d), want, 1e-3, 1e-4)
    silu_of_negated = -want / (1 + np.exp(want))
    orc.assert_close(run(ctx, x, wt, d=d, ops=(capi.UNARY_NEG, capi.UNARY_SILU)), silu_of_negated, 1e-3, 1e-4)
    wt.free()


@pytest.mark.parametrize("fmt,m,k,n", [(Q4, 65, 1024, 30005), (Q4, 300, 1024, 14369), (Q8, 65, 512, 50017)])
def test_two_streams_that_store_the_result_themselves(ctx, orc, fmt, m, k, n):
    """Each stream finishes one of a wave's two column tiles: residual, unary operations and a last column
    group whose tiles end inside or behind the result."""
    plan = capi.matmul_block_plan(fmt, m, k, n)
    assert plan.threads == 512 and plan.rows < 128 and plan.k_parts == 1
    w = synth.normal(2013, k * n, 0.02).reshape(k, n)
    x, d = synth.normal(2014, m * k).reshape(m, k), synth.normal(2015, m * n).reshape(m, n)
    wt = ctx.weight(fmt, w)
    want = x.astype(np.float64) @ orc.dequantize(fmt, orc.quantize(fmt, w), k, n).astype(np.float64)
    got = run(ctx, x, wt)
    assert_rows_close(got, want, x, k)
    added = run(ctx, x, wt, d=d)
    assert np.array_equal(added, got + d)
    assert np.array_equal(run(ctx, x, wt, d=d, ops=(capi.UNARY_NEG, capi.UNARY_RELU)), np.maximum(-added, 0))
    want += d
    orc.assert_close(run(ctx, x, wt, d=d, ops=(capi.UNARY_NEG, capi.UNARY_SILU)), -want / (1 + np.exp(want)), 1e-3, 1e-4)
    wt.free()


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("k", [1280, 4128])
def test_magnitudes_that_change_along_k(ctx, orc, fmt, k):
    """A row whose slices of 256 elements lie up to 2^70 apart keeps its relative accuracy where only the
    small slices meet a weight: the large slices' columns of the weight are zero blocks in the last column."""
    m, n = 35, 130
    w = synth.normal(2020, k * n, 0.02).reshape(k, n)
    w[:512, n - 1] = 0.0
    x = synth.normal(2021, m * k).reshape(m, k)
    x[3, 256:] *= np.float32(2.0**-30)
    x[4, 512:] *= np.float32(2.0**-70)
    x[5] *= np.float32(1e-25)
    x[6] *= np.float32(1e20)
    x[7, 300:700] = 0.0
    wt = ctx.weight(fmt, w)
    dq = orc.dequantize(fmt, orc.quantize(fmt, w), k, n)
    want = np.asarray(orc.matmul_f64(x, dq), np.float64)
    got = run(ctx, x, wt)
    assert_rows_close(got, want, x, k)
    small = np.abs(x[[3, 4]][:, 512:]).max(axis=1)
    assert (dq[:512, n - 1] == 0).all()
    err = np.abs(got[[3, 4], n - 1] - want[[3, 4], n - 1])
    assert (err <= 8 * 2.0**-21 * 0.06 * np.sqrt(k) * small).all(), err / small
    # infinities, NaNs and magnitudes of 2^100 stay in their rows
    y = x.copy()
    y[0, 5], y[1, 700], y[2, 40] = np.inf, np.nan, np.float32(2.0**101)
    bad = run(ctx, y, wt)
    assert not np.isfinite(bad[:3]).any()
    assert np.array_equal(bits(bad[3:]), bits(got[3:]))
    wt.free()


@pytest.mark.parametrize("fmt", [Q4, Q8])
def test_small_slices_beside_a_large_one(ctx, orc, fmt):
    """A slice of 256 elements keeps 22 bits of its own largest magnitude whatever the row's largest is, 2^14 (where the
    row's scale is 1) and its neighbours among them: seen in a column whose weights are zero over the large slice."""
    k, n = 1280, 130
    rows = [(top, small) for top in (2.0**13, 9000.0, 2.0**14, 20000.0, 32767.0, 2.0**15, 40000.0, 1.5, 1e-6, 1e9) for small in (2.0**-15, 2.0**-22, 2.0**-30, 2.0**-40)]
    m = len(rows)
    w = synth.normal(2060, k * n, 0.02).reshape(k, n)
    w[:256, n - 1] = 0.0
    x = synth.normal(2061, m * k).reshape(m, k)
    x /= np.abs(x).reshape(m, -1, 256).max(axis=2).repeat(256, axis=1)
    for r, (top, small) in enumerate(rows):
        x[r] *= np.float32(top)
        x[r, 256:] *= np.float32(small)
    wt = ctx.weight(fmt, w)
    dq = orc.dequantize(fmt, orc.quantize(fmt, w), k, n).astype(np.float64)
    assert (dq[:256, n - 1] == 0).all()
    want, got = x.astype(np.float64) @ dq, run(ctx, x, wt)
    assert_rows_close(got, want, x, k)
    assert_rows_close(got[:, n - 1:], want[:, n - 1:], x[:, 256:], k)
    wt.free()


@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("gap", [0, 3, 4, 7, 8, 12, 16])
def test_small_elements_of_a_slice(ctx, orc, fmt, gap):
    """Inside a slice 2^gap below the row's largest: elements far below the slice's own largest are held down to 2^-31 (Q4) or
    2^-35 (Q8) of that largest, as in the tiled kernels, and rounded, not cut.  The large elements meet blocks of zero
    weights and all products are positive, so that what every element loses adds up."""
    m, k, n = 33, 512, 70
    x = np.abs(synth.normal(2070, m * k)).reshape(m, k).astype(np.float32) + np.float32(0.5)
    x *= np.float32(2.0 ** (-gap - 20))
    x[:, :256] *= np.float32(2.0**20)
    x[:, 5], x[:, 261] = 1.0, 2.0**-gap
    w = np.abs(synth.normal(2071, k * n, 0.02)).reshape(k, n) + np.float32(0.001)
    w[:288] = 0.0
    x[:, :256] = np.minimum(x[:, :256], 1.0)
    wt = ctx.weight(fmt, w)
    dq = orc.dequantize(fmt, orc.quantize(fmt, w), k, n).astype(np.float64)
    assert (dq[:288] == 0).all() and (dq >= 0).all()
    want, got = x.astype(np.float64) @ dq, run(ctx, x, wt).astype(np.float64)
    held = 2.0 ** (-gap - (31 if fmt == Q4 else 35)) * dq.sum(axis=0)  # the last bit held of every element that meets a weight, of which it is half off at most
    # the f32 sums: 16 blocks and their means, 2^-24 each of the products' sum (Q8: of 128 scales per element, before the bias)
    biased = want if fmt == Q4 else (x[:, 288:].astype(np.float64).sum(axis=1) * 128)[:, None] * (dq.max(axis=0) / 127)
    assert (np.abs(got - want) <= held / 2 + 2.0**-20 * biased).all()
    wt.free()


@pytest.mark.parametrize("fmt", [Q4, Q8])
def test_activations_are_rounded_without_a_bias(ctx, orc, fmt):
    """The pairs that f32 activations enter as are rounded to nearest: over many outputs the errors have no part along the result
    (cut to 22 bits they have one of 2^-24 to 2^-23)."""
    m, k, n = 65, 4096, 513
    w = synth.normal(2080, k * n, 0.02).reshape(k, n)
    x = synth.normal(2081, m * k).reshape(m, k)
    wt = ctx.weight(fmt, w)
    want = x.astype(np.float64) @ orc.dequantize(fmt, orc.quantize(fmt, w), k, n).astype(np.float64)
    err = run(ctx, x, wt) - want
    # errors of at most 2^-19 of the result's size (8 x 2^-22), independent over m n outputs, average out to 2^-19 / sqrt(m n)
    assert abs((err * want).sum() / (want * want).sum()) <= 2.0**-26 + 2.0**-19 / np.sqrt(m * n)
    wt.free()


def test_q8_sums_are_free_of_the_byte_bias(ctx, orc):
    """Q8 with f32 activations that have a mean: a bias of 128 on the bytes would put sums of some hundred times the result's
    size into the accumulators.  Without one the error is that of the f32 additions, one per block of 32, each 2^-24
    of a sum no larger than the result's size, independent of each other."""
    m, k, n = 65, 4096, 513
    w = synth.normal(2090, k * n, 0.02).reshape(k, n)
    x = synth.normal(2091, m * k).reshape(m, k) + np.float32(8.0)
    wt = ctx.weight(Q8, w)
    want = x.astype(np.float64) @ orc.dequantize(Q8, orc.quantize(Q8, w), k, n).astype(np.float64)
    err = run(ctx, x, wt) - want
    assert np.linalg.norm(err) <= 2.0**-24 * np.sqrt(k / 32) * np.linalg.norm(want)
    wt.free()


# (one for each workgroup, K in one part)
@pytest.mark.parametrize("m,n", [(134, 13028), (98, 12724), (130, 18829), (198, 17016), (387, 13986), (388, 19172)])
def test_q8_bias_leaves_a_sum_that_holds_it(ctx, orc, m, n):
    """Q8 with fp16 activations multiplies bytes with a bias of 128 and takes it out of the sum of each two blocks.  Integers for which every
    sum on the way fits 24 bits if it is taken out when the products (one tile's: all but the last) are in, and none does if
    it is taken out first: 2^23 a stage, at a running sum of -2^24 + 1.5 x 2^22 and odd."""
    k, base = 736, 499
    assert capi.matmul_block_plan(Q8, m, k, n, True).k_parts == 1
    rng = np.random.default_rng(7)
    w = rng.integers(-10, 11, (k, base))
    w[30::32], w[31::32] = 127, -127  # a block's scale is 1
    w[30:128:32] = -107
    w[:64], w[64:128] = np.where(w[:64] == -127, -127, -107), np.where(w[64:128] == -127, -127, -51)
    x = np.full((m, k), 1024)
    x[np.arange(m), np.arange(m) % 31] += 1  # meets -107: the sums are odd
    sums = np.cumsum((x[:, :, None] * w[None, :, :1]).reshape(m, -1, 32).sum(axis=2), axis=1)
    assert ((sums[:, 3:] > 2**22 - 2**24) & (sums[:, 3:] < 2**23 - 2**24) & (sums[:, 3:] % 2 == 1)).all()
    packed = orc.quantize(Q8, w.astype(np.float32))
    assert np.array_equal(orc.dequantize(Q8, packed, k, base), w)
    wt = ctx.weight(Q8, np.ascontiguousarray(w.astype(np.float32)[:, np.arange(n) % base]))
    got = run(ctx, x.astype(np.float16), wt, True)
    assert np.array_equal(got, (x @ w).astype(np.float32)[:, np.arange(n) % base])
    wt.free()


# One, two and three blocks in K's last 128 elements (two halves of a Q4 stage), in the first stage and in later ones, whose ring slots wrap
@pytest.mark.parametrize("fmt", [Q4, Q8])
@pytest.mark.parametrize("m,k,n", [(40, 96, 70), (40, 160, 70), (70, 448, 130), (97, 704, 300), (300, 576, 1000), (260, 1248, 500)])
def test_infinite_rows_of_fp16_activations_stay_on_their_own(ctx, orc, fmt, m, k, n):
    """K ends inside the elements that are loaded at once: what lies behind a row's end is the beginning of the next."""
    x = synth.normal(2030, m * k).reshape(m, k).astype(np.float16)
    wt = ctx.weight(fmt, synth.normal(2031, k * n, 0.02).reshape(k, n))
    clean = run(ctx, x, wt, True)
    x[11, 0], x[12, 1] = np.inf, np.nan
    got = run(ctx, x, wt, True)
    rest = [r for r in range(m) if r not in (11, 12)]
    assert np.array_equal(bits(got[rest]), bits(clean[rest])) and not np.isfinite(got[[11, 12]]).any()
    wt.free()


def test_rows_beyond_the_workspace_run_in_blocks(ctx, orc):
    m, k, n = 2500, 16384, 64
    assert capi.matmul_block_plan(Q4, m, k, n).launches > 1
    w = synth.normal(2040, k * n, 0.02).reshape(k, n)
    x = np.tile(synth.normal(2041, 50 * k).reshape(50, k), (m // 50, 1))
    wt = ctx.weight(Q4, w)
    got = run(ctx, x, wt)
    want = np.asarray(orc.matmul_f64(x[:50], orc.dequantize(Q4, orc.quantize(Q4, w), k, n)), np.float64)
    for r in range(0, m, 50):
        assert_rows_close(got[r:r + 50], want, x[:50], k)
    wt.free()


# Parts that do not share evenly between the two streams of a workgroup: an odd number of stages, a shorter last part,
# one of a single stage (the second stream has none)
@pytest.mark.parametrize("fmt,m,k,n", [(Q4, 97, 3168, 9846), (Q4, 65, 3872, 11916), (Q4, 34, 4160, 14866), (Q8, 66, 3616, 6605), (Q8, 65, 2368, 8403),
                                       (Q8, 66, 2624, 10815)])
def test_two_streams(ctx, orc, fmt, m, k, n):
    plan = capi.matmul_block_plan(fmt, m, k, n)
    assert (plan.threads, plan.cols, plan.rows) == (512, 256, 96 if fmt == Q8 or m == 65 else 64) and plan.k_parts > 1
    w = synth.normal(2050, k * n, 0.02).reshape(k, n)
    w[:256, n - 1] = w[tail_slice(k):, n - 2] = 0.0
    x = synth.normal(2051, m * k).reshape(m, k)
    small = mixed_rows(x)
    wt = ctx.weight(fmt, w)
    dq = orc.dequantize(fmt, orc.quantize(fmt, w), k, n).astype(np.float64)
    want = x.astype(np.float64) @ dq
    got = run(ctx, x, wt)
    assert_rows_close(got, want, x, k)
    assert_small_slices(got, want, x, dq, small, n - 1, n - 2)
    assert np.array_equal(bits(run(ctx, x, wt)), bits(got)), "not repeatable"
    wt.free()


# Every workgroup that is built, with K in one part and in several, at ragged sizes for which the planner takes it:
# rows x columns x threads, then shape and parts
WORKGROUPS = {
    (Q4, False): [(32, 256, 256, 66, 1056, 17126, 1), (32, 256, 256, 67, 4320, 1278, 17), (64, 128, 256, 49, 736, 16625, 1), (64, 128, 256, 34, 6304, 858, 25),
                  (64, 256, 256, 387, 736, 16657, 1), (64, 256, 256, 34, 4128, 7231, 17), (64, 256, 512, 100, 1056, 16512, 1), (64, 256, 512, 67, 30496, 797, 30),
                  (96, 256, 256, 271, 736, 20163, 1), (96, 256, 256, 67, 4320, 3623, 17), (96, 256, 512, 233, 928, 18803, 1), (96, 256, 512, 67, 27808, 1552, 28),
                  (128, 256, 512, 296, 736, 19594, 1), (128, 256, 512, 197, 3232, 3273, 9), (192, 256, 512, 583, 736, 13585, 1), (192, 256, 512, 130, 4192, 5476, 11),
                  (256, 256, 512, 577, 160, 19639, 1), (256, 256, 512, 195, 3360, 8220, 7)],
    (Q4, True): [(32, 256, 256, 129, 96, 14369, 1), (32, 256, 256, 35, 2080, 16322, 2), (64, 128, 256, 905, 736, 2063, 1), (64, 128, 256, 34, 17440, 4091, 23),
                 (64, 256, 256, 395, 736, 16800, 1), (64, 256, 256, 34, 19488, 4016, 31), (96, 256, 256, 199, 736, 18696, 1), (96, 256, 256, 66, 15136, 3658, 17),
                 (128, 256, 512, 298, 736, 19605, 1), (128, 256, 512, 98, 12064, 4022, 16), (192, 256, 512, 583, 736, 13572, 1), (192, 256, 512, 163, 15840, 2549, 25),
                 (256, 256, 512, 523, 160, 21043, 1), (256, 256, 512, 195, 17504, 2638, 23)],
    (Q8, False): [(32, 256, 256, 51, 736, 16442, 1), (32, 256, 256, 39, 1568, 78, 25), (64, 128, 256, 167, 736, 10856, 1), (64, 128, 256, 34, 6880, 1109, 27),
                  (64, 256, 256, 115, 736, 16405, 1), (64, 256, 256, 34, 6112, 1565, 32), (96, 256, 256, 161, 160, 21882, 1), (96, 256, 256, 68, 3232, 3691, 17),
                  (96, 256, 512, 203, 736, 16738, 1), (96, 256, 512, 67, 14368, 1293, 29), (128, 256, 512, 326, 736, 16423, 1), (128, 256, 512, 100, 2272, 5405, 9),
                  (192, 256, 512, 400, 736, 18702, 1), (192, 256, 512, 132, 6240, 2323, 25), (256, 256, 512, 484, 160, 21765, 1), (256, 256, 512, 194, 1568, 10874, 5)],
    (Q8, True): [(32, 256, 256, 134, 736, 13028, 1), (64, 128, 256, 98, 736, 12724, 1), (64, 128, 256, 35, 8224, 6463, 10), (64, 256, 256, 130, 736, 18829, 1),
                 (64, 256, 256, 35, 11872, 3790, 17), (96, 256, 256, 198, 736, 17016, 1), (96, 256, 256, 66, 18016, 1977, 32), (128, 256, 512, 387, 736, 13986, 1),
                 (128, 256, 512, 99, 13088, 2805, 23), (192, 256, 512, 388, 736, 19172, 1), (192, 256, 512, 130, 9568, 3691, 17)],
}


@pytest.mark.parametrize("fmt,f16,rows,cols,threads,m,k,n,parts", [kind + shape for kind, shapes in WORKGROUPS.items() for shape in shapes])
def test_every_workgroup(ctx, orc, fmt, f16, rows, cols, threads, m, k, n, parts):
    """Products, rows of mixed scale, infinite and NaN rows beside the others, residuals and epilogues.  The weight's columns
    repeat after 1499 (no multiple of a tile), so that all outputs have a reference."""
    plan = capi.matmul_block_plan(fmt, m, k, n, f16)
    assert (plan.taken, plan.rows, plan.cols, plan.threads, plan.k_parts) == (1, rows, cols, threads, parts)
    base = min(n, 1499)
    w = synth.normal(2100, k * base, 0.02).reshape(k, base)
    x = synth.normal(2101, m * k).reshape(m, k)
    mixed = not f16 and k >= 512
    if mixed:
        w[:256, 5] = w[tail_slice(k):, 7] = 0.0
        small = mixed_rows(x)
    x = x.astype(np.float16) if f16 else x
    wide = np.ascontiguousarray(w[:, np.arange(n) % base])
    wt = ctx.weight(fmt, wide)
    del wide
    dq = orc.dequantize(fmt, orc.quantize(fmt, w), k, base).astype(np.float64)
    want = (x.astype(np.float64) @ dq)[:, np.arange(n) % base]
    got = run(ctx, x, wt, f16)
    assert_rows_close(got, want, x.astype(np.float32), k)
    if mixed:
        assert_small_slices(got, want, x, dq, small, 5, 7)
    # Rows that are not finite, among them some that begin so, which the row in front reads behind its end where K fills no
    # whole stage: inside a row tile, in the first row of one, at the far end of what is read
    y = x.copy()
    behind = max(1, -k % (128 if fmt == Q4 else 64))
    y[0, 0], y[1, k - 1], y[5, 0], y[32, 1], y[m - 1, behind - 1] = np.inf, np.nan, np.inf, np.nan, np.inf
    bad = run(ctx, y, wt, f16)
    hit = np.isin(np.arange(m), (0, 1, 5, 32, m - 1))
    assert not np.isfinite(bad[hit]).any() and np.array_equal(bits(bad[~hit]), bits(got[~hit]))
    d = synth.normal(2102, m * n).reshape(m, n)
    added = run(ctx, x, wt, f16, d=d)
    assert np.array_equal(added, got + d)
    if not f16:
        assert np.array_equal(run(ctx, x, wt, d=d, ops=(capi.UNARY_NEG, capi.UNARY_RELU)), np.maximum(-added, 0))
    wt.free()


def test_every_workgroup_is_in_the_list():
    source = open(os.path.join(os.path.dirname(capi.__file__), "csrc", "kernels_block.hip")).read()
    built = set()
    for fmt, f32, numbers in re.findall(r"block_config<([01]), (true|false), ([0-9, ]+)>\(", source):
        rt, wm, wn, _, _, _, wk = [int(v) for v in (numbers + ", 1").split(",")][:7]
        built.add((int(fmt), f32 == "false", 32 * rt * wm, 64 * wn, 64 * wm * wn * wk))
    assert built == {kind + shape[:3] for kind, shapes in WORKGROUPS.items() for shape in shapes} and len(built) == 30


@pytest.mark.parametrize("fmt,f16", [(Q4, False), (Q4, True), (Q8, False), (Q8, True)])
def test_results_that_pass_the_caches_by(ctx, orc, fmt, f16):
    """Just over 64 MiB of result, twice the chip's L2s, ragged in rows and columns.  Rows repeat after 41 and columns after 1499, so that all outputs
    have a reference."""
    m, k, n = 1025, 96, 16389
    assert m * n * 4 > 64 << 20 and capi.matmul_block_plan(fmt, m, k, n, f16).k_parts == 1
    w = synth.normal(2200, k * 1499, 0.02).reshape(k, 1499)
    base = synth.normal(2201, 41 * k).reshape(41, k).astype(np.float16 if f16 else np.float32)
    rows, cols = np.arange(m) % 41, np.arange(n) % 1499
    wt = ctx.weight(fmt, np.ascontiguousarray(w[:, cols]))
    want = base.astype(np.float64) @ orc.dequantize(fmt, orc.quantize(fmt, w), k, 1499).astype(np.float64)
    got = run(ctx, base[rows], wt, f16)
    # (not bit for bit across tiles: a wave's last tile adds a block's product behind the next blocks' means)
    assert_rows_close(got, want[rows][:, cols], base[rows].astype(np.float32), k)
    d = synth.normal(2202, m * n).reshape(m, n)
    assert np.array_equal(run(ctx, base[rows], wt, f16, d=d), got + d)
    wt.free()
