"""Sums of one to eight trees and products of one to three at every order
(the sum and the product kernels of a level) against the oracle's restatement.

Bar: identical node sets; coefficients within 1e-14 relative L2, as for the
two-operand cases.  A sum of eight accumulates 8 rounded products, a product of
three takes 3 (k+1)-term sums per direction per operand: both stay below 40
roundings of 1.1e-16 in the root mean square.  The value of a small factor carries
the rounding of its node's largest, so a product is only as accurate as its factors
overlap: exp(-b1 b2 / (b1 + b2) d^2) >= exp(-3 * 0.75) = 0.1 for the centers and
exponents here (narrow factors further apart, of overlap 1e-4, reach 1.2e-14).
"""
from math import erf

import numpy as np
import pytest

from mrcpp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [3, 5, 7, 9])
def test_sums_and_products_of_every_order(mr, orc, order):
    mra, omra = mr.MultiResolutionAnalysis((-8, 8), order), orc.OracleMRA((-8, 8), order)
    prec = 10.0 ** -(order // 2 + 1)
    pairs = []
    mr.set_projection_target("host")
    try:
        for s in range(3):
            src = W.random_sources(20 + s, 1 + s, center_range=0.25, beta_range=(1.0, 6.0))
            f = mr.FunctionTree(mra)
            gx = mr.GaussExp.from_sources(src)
            mr.build_grid(f, gx)
            mr.project(prec, f, gx)
            of = orc.OracleTree(omra)
            of.project_gaussians(prec, src.coefs, src.exponents, src.centers)
            pairs.append((f, of))
    finally:
        mr.set_projection_target("auto")

    def check(mine, ref):
        (mi, mc, mn), (oi, oc, on) = mine.export(), ref.export()
        assert np.array_equal(mi, oi)
        assert np.linalg.norm(mc - oc) <= 1e-14 * np.linalg.norm(oc)
        assert np.allclose(mn, on, rtol=1e-12, atol=1e-14 * max(1.0, np.abs(on).max()))

    for count in (1, 2, 8):
        terms = [(0.5 + 0.25 * i, pairs[i % 3]) for i in range(count)]
        h, oh = mr.FunctionTree(mra), orc.OracleTree(omra)
        mr.add(prec, h, [(c, p[0]) for c, p in terms])
        orc.add(prec, oh, [(c, p[1]) for c, p in terms])
        check(h, oh)
    for count in (1, 2, 3):
        terms = [(1.5 - 0.25 * i, pairs[i]) for i in range(count)]
        h, oh = mr.FunctionTree(mra), orc.OracleTree(omra)
        mr.multiply(prec, h, [(c, p[0]) for c, p in terms])
        orc.multiply(prec, oh, [(c, p[1]) for c, p in terms])
        check(h, oh)


@pytest.mark.parametrize("order", [3, 5, 7, 9])
@pytest.mark.parametrize("beta,distance", [(3.0, 0.4), (20.0, 0.8), (20.0, 1.1), (60.0, 0.6), (200.0, 0.5)])
def test_product_of_factors_far_apart(mr, orc, order, beta, distance):
    """Two narrow Gaussians of overlap 0.8 down to 1e-11: the product is far
    smaller than its factors and the order of the sums shows (relative to the
    product up to 4e-10).  In a node a value of f carries the rounding of f's norm
    there over the square root of the volume, and so the product that of both
    norms: with 18 passes (six of either factor, six back), each rounding by
    less than two units in the last place, the end nodes differ by at most
    36 2^-53 sqrt(sum_n (|f|_n |g|_n)^2 / vol_n)."""
    mra, omra = mr.MultiResolutionAnalysis((-8, 8), order), orc.OracleMRA((-8, 8), order)
    prec = 10.0 ** -(order // 2 + 1)
    centers = [(0.1 + s * distance / 2, 0.05, -0.02) for s in (-1, 1)]
    mine, ref, gauss = [], [], []
    mr.set_projection_target("host")
    try:
        for c in centers:
            src = W.GaussianSources([1.0], [beta], [c])
            gx = mr.GaussExp.from_sources(src)
            f = mr.FunctionTree(mra)
            mr.build_grid(f, gx)
            mr.project(prec, f, gx)
            of = orc.OracleTree(omra)
            of.project_gaussians(prec, src.coefs, src.exponents, src.centers)
            mine.append((1.0, f))
            ref.append((1.0, of))
            gauss.append(gx.funcs[0])
    finally:
        mr.set_projection_target("auto")
    h, oh = mr.FunctionTree(mra), orc.OracleTree(omra)
    mr.multiply(prec, h, mine)
    orc.multiply(prec, oh, ref)
    (mi, mc, _), (oi, oc, _) = h.export(), oh.export()
    assert np.array_equal(mi, oi)
    end = mi[:, 4] == 1
    size = mra.scaling_factor * 2.0 ** -mi[end, 0].astype(float)
    lo = size[:, None] * mi[end, 1:4]
    norms = size ** -1.5
    for g in gauss:
        a = np.sqrt(2.0 * g.alpha)
        e = np.vectorize(erf)(a * (lo + size[:, None] - g.pos)) - np.vectorize(erf)(a * (lo - g.pos))
        norms = norms * abs(g.coef) * np.sqrt(np.prod(np.sqrt(np.pi) / (2.0 * a) * e, axis=1))
    err = np.linalg.norm(mc[end] - oc[end])
    print("case", order, beta, distance, "nodes", len(mi), "relative", err / np.linalg.norm(oc[end]), "of the bar", err / (36 * 2.0 ** -53 * np.linalg.norm(norms)))
    assert err <= 36 * 2.0 ** -53 * np.linalg.norm(norms)
