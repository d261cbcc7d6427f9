"""A session's launches of more than four rows that serve several weights or take a norm or a SwiGLU along: the same
step with launch fusion on and off (the general path: one dispatch, one launch), at the edges of row groups,
slices, K parts and column groups, with every kind of row that the conversion treats apart."""
import numpy as np
import pytest

from helpers import Q8
from meganeura_amd import capi, synth
from meganeura_amd.graph import Graph, build_inference_session

pytestmark = pytest.mark.gpu


def rows_of(m, k, seed):
    """Activations of ordinary size, with rows of zeros, of tiny and of large values and of slices far apart."""
    x = synth.normal(seed, m * k).reshape(m, k).copy()
    x[0] = 0
    x[m // 2] *= 1e-12
    x[m - 1] *= 1e9
    x[m - 2, : k // 2] *= 1e-4
    return x


def step_outputs(sess, sizes):
    sess.step()
    sess.wait()
    return [sess.read_output_by_index(i, s) for i, s in enumerate(sizes)]


def close(a, b, m, bound):
    """Row by row: the same products and the same sums but for the order of the norm's and of K parts
    that a joint plan may cut elsewhere: f32 sums over at most 4096 terms, 2^-24 sqrt(4096) = 4e-6 of the row's size,
    and the activations' 2^-22 behind a norm that differs by that."""
    a, b = a.reshape(m, -1).astype(np.float64), b.reshape(m, -1).astype(np.float64)
    assert np.isfinite(a).all()
    err, size = np.linalg.norm(a - b, axis=1), np.linalg.norm(b, axis=1)
    assert (err <= bound * size + 1e-30).all(), (err / np.maximum(size, 1e-30)).max()


def layer(quant, m, k, cols, with_norm, residual):
    g = Graph()
    x = g.input("x", [m, k])
    a = g.rms_norm(x, g.parameter("norm", [k]), 1e-5) if with_norm else x
    outs = []
    for i, n in enumerate(cols):
        y = g.matmul(a, (g.parameter_q4 if quant == "q4" else g.parameter_q8)(f"w{i}", [k, n]))
        outs.append(g.add(y, g.input(f"r{i}", [m, n])) if residual else y)
    g.set_outputs(outs)
    s = build_inference_session(g)
    s.set_input("x", rows_of(m, k, m + k))
    if with_norm:
        s.set_parameter("norm", 1.0 + 0.1 * synth.normal(5, k))
    for i, n in enumerate(cols):
        s.set_parameter(f"w{i}", synth.normal(10 + i, k * n, 0.02))
        if residual:
            s.set_input(f"r{i}", synth.normal(20 + i, m * n))
    return s


@pytest.mark.parametrize("quant", ["q4", "q8"])
@pytest.mark.parametrize("m,k,cols,norm,residual,launches", [
    (128, 1024, (1024, 512, 512), True, False, (1, 1)),  # q | k | v behind their norm
    (333, 1024, (1024, 512, 512), True, False, (1, 1)),
    (129, 288, (100, 31, 517), True, True, (1, 1)),  # ragged columns, a slice and a bit of K, residuals
    (145, 32, (1, 16, 15), True, False, (1, 1)),  # one block of K
    (128, 1024, (256, 257), False, True, (1, 1)),  # no norm; a column group of one column
    (128, 1056, (300, 64, 64), True, False, (2, 4)),  # K in two parts: the norm stays its own launch
    (130, 2080, (128, 96), False, True, (1, 1)),  # three K parts
    (512, 1024, (512, 512), True, False, (1, 1)),  # whether one round or not
    (24, 576, (576, 192, 192), True, False, (1, 1)),
    (7, 1024, (192, 64), True, True, (1, 1)),
    (20, 544, (33, 257, 16), True, True, (1, 1)),
    (160, 1024, (515, 100, 31), True, True, (1, 1)),
    (17, 1056, (300, 64, 64), True, True, (2, 4)),
    (31, 2080, (128, 96), False, True, (1, 1)),
])
def test_several_weights_behind_a_norm(quant, m, k, cols, norm, residual, launches):
    s = layer(quant, m, k, cols, norm, residual)
    sizes = [m * n for n in cols]
    assert s.num_launches() == launches[quant == "q8"]  # (Q4, Q8): a weight that another kernel takes keeps its launch
    fused = step_outputs(s, sizes)
    again = step_outputs(s, sizes)
    s.set_graph_replay(True)
    replayed = [step_outputs(s, sizes) for _ in range(4)][-1]
    s.set_graph_replay(False)
    s.set_fusion(False)
    plain = step_outputs(s, sizes)
    s.close()
    for f, a, r, p in zip(fused, again, replayed, plain):
        assert np.array_equal(f, a) and np.array_equal(f, r)
        close(f, p, m, 1e-5)


@pytest.mark.parametrize("quant", ["q4", "q8"])
@pytest.mark.parametrize("m,k,n,residual,launches", [(128, 1024, 512, True, (2, 2)), (333, 3072, 1024, True, (2, 2)), (129, 288, 100, False, (2, 2)), (145, 1056, 17, True, (2, 3)),
                                            (16, 1536, 576, True, (2, 2)), (5, 2048, 64, False, (2, 2))])
def test_swiglu_on_the_way(quant, m, k, n, residual, launches):
    g = Graph()
    par = g.parameter_q4 if quant == "q4" else g.parameter_q8
    x = g.input("x", [m, 64])
    gate, up = g.matmul(x, par("wg", [64, k])), g.matmul(x, par("wu", [64, k]))
    y = g.matmul(g.swiglu(gate, up), par("wd", [k, n]))
    if residual:
        y = g.add(y, g.input("r", [m, n]))
    g.set_outputs([y])
    s = build_inference_session(g)
    s.set_input("x", synth.normal(1, m * 64))
    for i, (name, count) in enumerate((("wg", 64 * k), ("wu", 64 * k), ("wd", k * n))):
        s.set_parameter(name, synth.normal(30 + i, count, 0.1))
    if residual:
        s.set_input("r", synth.normal(40, m * n))
    assert s.num_launches() == launches[quant == "q8"]
    fused = step_outputs(s, [m * n])[0]
    s.set_fusion(False)
    plain = step_outputs(s, [m * n])[0]
    s.close()
    close(fused, plain, m, 1e-5)


@pytest.mark.parametrize("m,k,n", [(33, 32, 1), (47, 288, 257), (64, 1056, 70), (127, 4096, 300), (96, 3584, 513), (113, 2080, 1025)])
def test_q8_of_33_to_127_rows(orc, m, k, n):
    """The automatic choice against 64 bits; every product carries 22 bits of the row's largest slice and sums are f32:
    8 (2^-22 + 2^-24) sqrt(K) of the row's largest magnitude times the weights' size (0.02, zero points included 0.06)."""
    w, x, d = synth.normal(60, k * n, 0.02).reshape(k, n), rows_of(m, k, 61), synth.normal(62, m * n).reshape(m, n)
    dq = orc.dequantize(Q8, orc.quantize(Q8, w), k, n).astype(np.float64)
    with capi.Context(0) as ctx:
        wt, a, c, dd = ctx.weight(Q8, w), ctx.upload(x), ctx.buffer(m * n * 4), ctx.upload(d)
        bound = 8 * (2.0**-22 + 2.0**-24) * 0.06 * np.sqrt(k) * np.abs(x).max(axis=1, keepdims=True).astype(np.float64)
        for res in (None, dd):
            ctx.matmul_q(a, wt, c, m, res)
            got = c.download(np.float32, m * n).reshape(m, n)
            want = x.astype(np.float64) @ dq + (d if res else 0)
            assert (np.abs(got - want) <= bound + 2.0**-23 * np.abs(want)).all()
            ctx.matmul_q(a, wt, c, m, res)
            assert np.array_equal(c.download(np.float32, m * n).reshape(m, n), got), "not repeatable"
        for b in (a, c, dd, wt):
            b.free()
