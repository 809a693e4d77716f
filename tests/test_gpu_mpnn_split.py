"""The network's products on split FP32 operands: remainders of the 128-row
tiles, and values that do not split (past the largest BF16, infinities, NaN),
which take the FP32 sums."""
import numpy as np
import pytest

import mpnn
import phenlei_amd as pa

pytestmark = pytest.mark.gpu


def chain(n):
    nbr = -np.ones((n, 2), np.int32)
    nbr[1:, 0] = np.arange(n - 1)
    nbr[:-1, 1] = np.arange(1, n)
    return nbr


def problem(n, layers=2, seed=0):
    rng = np.random.default_rng(seed)
    net = pa.Mpnn(layers=layers, seed=seed)
    p = net.get_params()
    for k in ("b0", "c", "bo"):
        p[k] = (0.05 * rng.standard_normal(p[k].shape)).astype(np.float32)
    net.set_params(p)
    net.set_graph(chain(n))
    X = rng.standard_normal((n, 8)).astype(np.float32)
    T = rng.standard_normal((n, 5)).astype(np.float32)
    net.set_data(X, T)
    return net, p, X, T, chain(n)


@pytest.mark.parametrize("n", [1, 2, 31, 127, 128, 129, 257, 700])
def test_rows_at_tile_edges(n):
    """FP32 rounding of sums of 256 products and six layers of them stays
    well inside 1e-5 (forward) and 1e-4 (gradients) of the largest value, as
    for the oracle comparison at full tiles."""
    net, p, X, T, nbr = problem(n)
    p64 = {k: v.astype(np.float64) for k, v in p.items()}
    y, yr = net.forward(), mpnn.forward(p64, X.astype(np.float64), nbr)
    assert np.max(np.abs(y - yr)) <= 1e-5 * np.max(np.abs(yr))
    loss, g = net.gradient()
    lr, gr = mpnn.backward(p64, X.astype(np.float64), nbr, T.astype(np.float64))
    assert loss == pytest.approx(lr, rel=1e-5)
    for k in gr:
        assert np.max(np.abs(g[k] - gr[k])) <= 1e-4 * max(np.max(np.abs(gr[k])), 1e-30), k


def relu(z):
    return np.where(z > 0, z, np.float32(0))  # of a NaN: zero, as the kernels take it


@pytest.mark.parametrize("where", ["row", "weight"])
@pytest.mark.parametrize("value", [3.4e38, np.inf, np.nan])
def test_values_that_do_not_split(where, value):
    """One layer whose sums have one term each, a feature or a weight out of
    the splitting range: the result is numpy's in FP32, value for value (3.4e38
    times 2^-10 stays finite, an overflow is an infinity, an infinity times
    zero a NaN)."""
    n = 300
    net, p, X, T, nbr = problem(n, layers=1)
    for k in p:
        p[k][...] = 0
    p["W0"][0, 0] = 1.0
    p["A"][0, 0, 3] = 2.0 ** -10
    p["Wo"][3, 0] = 1.0
    X[...] = 0
    X[:, 0] = 1.0 + np.arange(n) % 7
    if where == "row":
        X[200, 0] = value
    else:
        p["A"][0, 0, 3] = value
    net.set_params(p)
    net.set_data(X, T)
    with np.errstate(invalid="ignore", over="ignore"):
        h = relu(X @ p["W0"])
        m = np.zeros_like(h)
        for i in range(n):
            js = nbr[i][nbr[i] >= 0]
            m[i] = h[js].sum(axis=0) * np.float32(1 / len(js))
        z = h @ p["A"][0] + m @ p["B"][0]
        want = (h + relu(z)) @ p["Wo"]
    assert np.array_equal(net.forward(), want, equal_nan=True)


@pytest.mark.parametrize("n,layers", [(8193, 6), (20011, 6), (70001, 3), (525000, 1)])
def test_gradients_over_several_slabs(n, layers):
    """Weight gradients are sums over chunks of rows, each staged in slabs of 32:
    two slabs with a last chunk of one row, three with a ragged end, chunks of
    288 rows (and of 69 for the edge layers), and the largest, 2,048 rows.
    Within 1e-4 of each gradient's largest value, as at the tiles' edges; a
    slab left out or taken twice would be off by about 1/sqrt(chunks) of it."""
    net, p, X, T, nbr = problem(n, layers=layers, seed=2)
    loss, g = net.gradient()
    lr, gr = mpnn.backward({k: v.astype(np.float64) for k, v in p.items()}, X.astype(np.float64), nbr,
                           T.astype(np.float64))
    assert loss == pytest.approx(lr, rel=1e-5)
    for k in gr:
        assert np.max(np.abs(g[k] - gr[k])) <= 1e-4 * np.max(np.abs(gr[k])), k


@pytest.mark.parametrize("big", [0, 1])
def test_weight_gradients_of_values_that_do_not_split(big):
    """Two rows, each the other's neighbour, only the first with a loss: A's
    gradient holds the row's own feature times dz, B's the neighbour's.  One
    of the two features is past the splitting range."""
    net, p, X, T, _ = problem(2, layers=1)
    for k in p:
        p[k][...] = 0
    p["W0"][0, 5] = 1.0
    p["c"][0, 9] = 1.0
    p["Wo"][9, 0] = 2.0 ** -10
    X[...] = 0
    X[:, 0] = (3.4e38, 3.0) if big == 0 else (3.0, 3.4e38)
    T[...] = 0
    T[1, 0] = 2.0 ** -10  # what the second row gives: z = 1, y = 2^-10
    net.set_params(p)
    net.set_data(X, T)
    g = net.gradient()[1]
    dz = np.float32(g["c"][0, 9])
    assert dz > 0 and g["c"][0].astype(bool).sum() == 1
    for name, x in (("A", X[0, 0]), ("B", X[1, 0])):
        want = np.zeros((128, 128), np.float32)
        want[5, 9] = x * dz
        assert np.allclose(g[name][0], want, rtol=2.0 ** -23, atol=0), name
