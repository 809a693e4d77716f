"""Single products of the network's dense layers and weight gradients against
64 bits.  Every sum here has one term that is not zero, so its value is one
product of two FP32 numbers.  The split form makes it of exact BF16 products:
the leading one, exact in the FP32 accumulator; five others, at most 2^-7 of it
in all, summed with at most six roundings of 2^-24 of their sum; one FP32
addition of the two (2^-24 of the product); and the three left out, at most
2 x 2^-25 + 2^-34 of it.  Its bound is therefore 2^-23 (1 + 2^-4) of the
product, where a product rounded to FP32 is within 2^-24."""
import numpy as np
import pytest

import phenlei_amd as pa

pytestmark = pytest.mark.gpu

BOUND = 2.0 ** -23 * (1 + 2.0 ** -4)
# splits into 1, 2^-8 and -2^-17, all of which are as large as they can be
EDGE = 1 + 2.0 ** -8 - 2.0 ** -17


def values(n, exponent, rng):
    """n FP32 numbers of [1, 2) 2^exponent, exact there too, some of them at the
    edges of the split (rounded to FP32's subnormal grain below 2^-126)."""
    v = rng.uniform(1.0, 2.0, n).astype(np.float32)
    v[:4] = EDGE, EDGE + 2.0 ** -23, 1 + 2.0 ** -8, 2 - 2.0 ** -23
    v[4:20] = (EDGE + 2.0 ** -18 * rng.uniform(-1, 1, 16)).astype(np.float32)
    return (v.astype(np.float64) * 2.0 ** exponent).astype(np.float32)


def check(got, want):
    got = np.asarray(got, np.float64)
    assert np.all(np.isfinite(got))
    err = np.max(np.abs(got - want) / want)
    print("relative error in units of 2^-24:", err * 2.0 ** 24)
    assert err <= BOUND


def zero_net():
    net = pa.Mpnn(layers=1, seed=0)
    p = net.get_params()
    for k in p:
        p[k][...] = 0
    return net, p


def forward_products(v, w):
    """v_i w_j by the hidden layer's forward product: h[i][0] = v_i,
    A[0][3 + j] = w_j."""
    net, p = zero_net()
    p["W0"][0, 0] = 1.0
    for j in range(5):
        p["A"][0, 0, 3 + j] = w[j]
        p["Wo"][3 + j, j] = 1.0
    net.set_params(p)
    net.set_graph(-np.ones((len(v), 1), np.int32))
    X = np.zeros((len(v), 8), np.float32)
    X[:, 0] = v
    net.set_data(X)
    return net.forward()


def gradient_products(v, a, scale, which):
    """Two rows that are each other's neighbour, with the same h = v; only the
    first has a loss, so dz has one row, whose values c's gradient gives.
    Returns (dz, gradient of A, gradient of B, gradient of b0): of A and of B
    v_k dz_j, of b0 a_k dz_0 (which: through A^T or through B^T)."""
    K = len(v)
    net, p = zero_net()
    p["b0"][:K] = v
    p["c"][0, 120:125] = 1.0
    p[which][0, :K, 120] = a
    rng = np.random.default_rng(5)
    for j in range(5):
        p["Wo"][120 + j, j] = np.float32(rng.uniform(1, 2)) * np.float32(2.0) ** scale
    net.set_params(p)
    net.set_graph(np.array([[1], [0]], np.int32))
    X = np.zeros((2, 8), np.float32)
    net.set_data(X, np.zeros((2, 5), np.float32))
    T = net.forward()
    T[0] -= np.float32(0.75) * np.maximum(np.abs(T[0]), 1)
    net.set_data(X, T)
    g = net.gradient()[1]
    dz = g["c"][0, 120:125].astype(np.float64)
    assert np.all(dz > 0)
    return dz, g["A"][0, :K, 120:125], g["B"][0, :K, 120:125], g["b0"][:K]


def test_forward_products():
    rng = np.random.default_rng(1)
    v, w = values(1000, 0, rng), values(24, 0, rng)[:5]
    check(forward_products(v, w), v[:, None].astype(np.float64) * w.astype(np.float64))


@pytest.mark.parametrize("which", ["A", "B"])
def test_gradient_products(which):
    rng = np.random.default_rng(2)
    v, a = values(110, 0, rng), values(110, 0, rng)
    dz, gA, gB, gb0 = gradient_products(v, a, 0, which)
    want = v[:, None].astype(np.float64) * dz
    check(gA, want)
    check(gB, want)
    check(gb0, a.astype(np.float64) * dz[0])


@pytest.mark.parametrize("exponent", [-95, -105, -110, -111, -118, -126, -135])
def test_products_of_tiny_values(exponent):
    """Values whose pieces are BF16 subnormals (from 2^-103 down) or do not hold
    all of them (below 2^-110), on either side of a product that FP32 holds."""
    rng = np.random.default_rng(3)
    tiny, large = values(300, exponent, rng), values(24, 60, rng)[:5]
    check(forward_products(tiny, large), tiny[:, None].astype(np.float64) * large.astype(np.float64))
    tiny, large = values(24, exponent, rng)[:5], values(300, 60, rng)
    check(forward_products(large, tiny), large[:, None].astype(np.float64) * tiny.astype(np.float64))
    for v, a, scale in ((exponent, 0, 60), (60, 0, exponent), (0, exponent, 60), (0, 60, exponent)):
        hv, av = values(110, v, rng), values(110, a, rng)
        for which in ("A", "B"):
            dz, gA, gB, gb0 = gradient_products(hv, av, scale, which)
            if v + scale > -100:
                check(gA, hv[:, None].astype(np.float64) * dz)
                check(gB, hv[:, None].astype(np.float64) * dz)
            if a + scale > -100:
                check(gb0, av.astype(np.float64) * dz[0])


@pytest.mark.parametrize("which", ["A", "B"])
def test_products_below_the_largest_fp32(which):
    """Products of up to 2^128 (1 - 2^-14): where the factors round up to BF16,
    the leading pieces' product is an infinity, the values' is not."""
    v = np.full(110, (2 - 2.0 ** -9) * 2.0 ** 63, np.float32)
    w = np.full(5, (2 - 2.0 ** -10) * 2.0 ** 63, np.float32)
    check(forward_products(v, w), v[:, None].astype(np.float64) * w.astype(np.float64))
    one, small, none = (np.full(110, x, np.float32) for x in (1.0, 2.0 ** -100, 0.0))
    dz = gradient_products(one, none, 62, which)[0]
    v = (2.0 ** 128 * (1 - np.arange(1, 111) * 2.0 ** -14) / dz.max()).astype(np.float32)
    dz, gA, gB, _ = gradient_products(v, none, 62, which)
    check(gA, v[:, None].astype(np.float64) * dz)
    check(gB, v[:, None].astype(np.float64) * dz)
    dz = gradient_products(small, one, 62, which)[0]
    v = (2.0 ** 128 * (1 - np.arange(1, 111) * 2.0 ** -14) / dz[0]).astype(np.float32)
    dz, _, _, gb0 = gradient_products(small, v, 62, which)
    check(gb0, v.astype(np.float64) * dz[0])
