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
