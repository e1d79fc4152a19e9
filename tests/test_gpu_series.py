"""GPU parity of the arithmetic, series product and polynomial eval/diff
kernels against the oracle and the reference's golden vectors.  The device
code follows the reference's operation order with fused two_prod, so every
result must be bit-identical."""
import os

import numpy as np
import pytest

from oraclelib import GOLDEN, oracle, pd, pi, rand_cmd, rand_md

pytestmark = pytest.mark.gpu

OPS = ["add", "sub", "mul", "div", "sqrt"]


@pytest.mark.parametrize("K", [2, 4, 8])
@pytest.mark.parametrize("op", range(5))
def test_md_batch_golden(K, op):
    from phcpack_amd.series import md_batch
    g = np.load(os.path.join(GOLDEN, "md_ops.npz"))
    a, b = g[f"a{K}"], g[f"b{K}"]
    if op == 4:
        a = np.ascontiguousarray(np.abs(a) * np.sign(a[0]))
    c = md_batch(op, K, a, b)
    assert np.array_equal(c, g[f"{OPS[op]}{K}"]), (K, op)


@pytest.mark.parametrize("K", [2, 4, 8])
def test_md_batch_random_vs_oracle(K):
    from phcpack_amd.series import md_batch
    rng = np.random.default_rng(21 + K)
    n = 4099
    a = rand_md(rng, K, (n,), -100, 100)
    b = rand_md(rng, K, (n,), -1, 1)
    for op in range(5):
        aa = np.ascontiguousarray(np.abs(a) * np.sign(a[0])) if op == 4 else a
        c = np.zeros((K, n))
        oracle().omd_batch(op, K, n, pd(aa), pd(b), pd(c))
        assert np.array_equal(md_batch(op, K, aa, b), c), (K, op)


@pytest.mark.parametrize("K", [1, 2, 4, 8])
@pytest.mark.parametrize("cplx", [0, 1])
def test_product_batch_vs_oracle(K, cplx):
    from phcpack_amd.series import product
    rng = np.random.default_rng(100 + K + cplx)
    for deg in (0, 8, 15, 31):
        nb = 37
        gen = (lambda s: rand_cmd(rng, K, s)) if cplx else (lambda s: rand_md(rng, K, s))
        x, y = gen((nb, deg + 1)), gen((nb, deg + 1))
        z = product(K, cplx, x, y)
        for b in range(nb):
            xb, yb = np.ascontiguousarray(x[:, b]), np.ascontiguousarray(y[:, b])
            zb = np.zeros_like(xb)
            oracle().osr_product(K, cplx, deg, pd(xb), pd(yb), pd(zb))
            assert np.array_equal(z[:, b], zb), (K, cplx, deg, b)


# both sides of each line of the rule for pairs of products: K*D at 63..64,
# K = 2 at 65536 coefficients, a row of 256 and 257, the LDS limit (D = 128 at
# complex octo-double, 129 not), blocks with idle lanes, odd and even batches,
# and signed zeros in double
@pytest.mark.parametrize("K,cplx,deg,nb", [(1, 0, 62, 3), (1, 0, 63, 3), (1, 1, 63, 4), (1, 0, 255, 5),
                                           (1, 0, 256, 5), (2, 0, 30, 2), (2, 1, 31, 1), (2, 1, 0, 65535),
                                           (2, 1, 8, 7281), (2, 1, 8, 7282), (4, 0, 14, 6), (4, 1, 42, 7),
                                           (8, 0, 7, 33), (8, 1, 127, 2), (8, 1, 128, 2)])
def test_product_pairs_vs_oracle(K, cplx, deg, nb):
    from phcpack_amd.series import product
    rng = np.random.default_rng(7 * deg + nb)
    gen = (lambda s: rand_cmd(rng, K, s)) if cplx else (lambda s: rand_md(rng, K, s))
    x, y = gen((nb, deg + 1)), gen((nb, deg + 1))
    if K == 1:
        x[:, :, 0] = -0.0
    z = product(K, cplx, x, y)
    for b in range(nb) if nb < 100 else (0, 1, nb // 2, nb - 2, nb - 1):
        xb, yb = np.ascontiguousarray(x[:, b]), np.ascontiguousarray(y[:, b])
        zb = np.zeros_like(xb)
        oracle().osr_product(K, cplx, deg, pd(xb), pd(yb), pd(zb))
        assert np.array_equal(z[:, b], zb) and np.array_equal(np.signbit(z[:, b]), np.signbit(zb)), b


@pytest.mark.parametrize("K", [2, 4, 8])
@pytest.mark.parametrize("cplx", [0, 1])
def test_product_golden(K, cplx):
    from phcpack_amd.series import product
    g = np.load(os.path.join(GOLDEN, "products.npz"))
    assert np.array_equal(product(K, cplx, g[f"x{K}_{cplx}"], g[f"y{K}_{cplx}"]),
                          g[f"z{K}_{cplx}"])


@pytest.mark.parametrize("K", [2, 4, 8])
@pytest.mark.parametrize("cplx", [0, 1])
def test_poly_evaldiff_golden(K, cplx):
    """Config-1 shape: 8 variables, 8 monomials of 3 variables, degree 15."""
    from phcpack_amd.series import PolyPlan
    g = np.load(os.path.join(GOLDEN, "poly.npz"))
    t = f"{K}_{cplx}"
    nvr, idx = g["nvr"], g["idx"]
    ptr = np.concatenate([[0], np.cumsum(nvr)])
    supports = [list(idx[ptr[i]:ptr[i + 1]]) for i in range(len(nvr))]
    plan = PolyPlan(K, cplx, 8, 15, supports, g["cst" + t], g["cff" + t])
    out = plan.evaldiff(g["inp" + t][:, None])
    assert np.array_equal(out[:, 0], g["out" + t])


def oracle_poly(K, cplx, nvr, idx, cst, cff, inp):
    P, dim, D = inp.shape
    ptr = np.concatenate([[0], np.cumsum(nvr)]).astype(np.int32)
    out = np.zeros((P, dim + 1, D))
    oracle().osr_poly_evaldiff(K, cplx, dim, len(nvr), D - 1, pi(nvr), pi(ptr), pi(idx),
                               pd(cst), pd(cff), pd(np.ascontiguousarray(inp)), pd(out))
    return out


@pytest.mark.parametrize("K", [1, 2, 4, 8])
@pytest.mark.parametrize("cplx", [0, 1])
def test_poly_evaldiff_batch_vs_oracle(K, cplx):
    """Random supports with 1..6 variables per monomial, a batch of inputs."""
    from phcpack_amd.series import PolyPlan
    rng = np.random.default_rng(300 + K * 2 + cplx)
    dim, nbr, deg, nb = 7, 10, 8, 19
    nvr = rng.integers(1, 7, nbr).astype(np.int32)
    supports = [sorted(rng.choice(dim, v, replace=False).tolist()) for v in nvr]
    idx = np.array([j for s in supports for j in s], np.int32)
    gen = (lambda s: rand_cmd(rng, K, s)) if cplx else (lambda s: rand_md(rng, K, s))
    cst, cff, inp = gen((deg + 1,)), gen((nbr, deg + 1)), gen((nb, dim, deg + 1))
    plan = PolyPlan(K, cplx, dim, deg, supports, cst, cff)
    out = plan.evaldiff(inp)
    for b in range(nb):
        assert np.array_equal(out[:, b], oracle_poly(K, cplx, nvr, idx, cst, cff, inp[:, b])), b


@pytest.mark.parametrize("K,cplx,deg,nb", [(2, 0, 0, 1), (1, 1, 1, 3), (4, 0, 32, 2), (2, 1, 63, 1),
                                           (2, 0, 64, 3), (8, 1, 40, 1), (4, 1, 6, 130)])
def test_poly_evaldiff_edges(K, cplx, deg, nb):
    """One coefficient, groups that do not fill a wavefront or need two, the
    operand rows in LDS and (K = 8) in global memory, monomials of 1..7
    variables in one polynomial."""
    from phcpack_amd.series import PolyPlan
    rng = np.random.default_rng(900 + 64 * K + deg)
    dim, nvr = 7, np.array([3, 1, 7, 2, 4, 1, 5, 6, 2], np.int32)
    supports = [sorted(rng.choice(dim, v, replace=False).tolist()) for v in nvr]
    idx = np.array([j for s in supports for j in s], np.int32)
    gen = (lambda s: rand_cmd(rng, K, s)) if cplx else (lambda s: rand_md(rng, K, s))
    cst, cff, inp = gen((deg + 1,)), gen((len(nvr), deg + 1)), gen((nb, dim, deg + 1))
    out = PolyPlan(K, cplx, dim, deg, supports, cst, cff).evaldiff(inp)
    for b in sorted({0, nb // 2, nb - 1}):
        assert np.array_equal(out[:, b], oracle_poly(K, cplx, nvr, idx, cst, cff, inp[:, b])), b


def test_poly_evaldiff_passes():
    """A batch whose contributions exceed the 256 MiB of one pass (here 62
    instances), against each instance alone; and a plan without monomials."""
    from phcpack_amd.series import PolyPlan
    rng = np.random.default_rng(17)
    K, dim, deg, nbr, nb = 8, 4, 16, 500, 130
    supports = [sorted(rng.choice(dim, 3, replace=False).tolist()) for _ in range(nbr)]
    cst, cff = rand_cmd(rng, K, (deg + 1,)), rand_cmd(rng, K, (nbr, deg + 1))
    inp = rand_cmd(rng, K, (nb, dim, deg + 1))
    plan = PolyPlan(K, 1, dim, deg, supports, cst, cff)
    out = plan.evaldiff(inp)
    for b in (0, 60, 61, 62, 123, 124, 129):
        assert np.array_equal(out[:, b:b + 1], plan.evaldiff(np.ascontiguousarray(inp[:, b:b + 1]))), b
    empty = PolyPlan(K, 1, dim, deg, [], cst, np.zeros((2 * K, 0, deg + 1))).evaldiff(inp[:, :2])
    assert np.array_equal(empty[:, 1, dim], cst) and not empty[:, :, :dim].any()
