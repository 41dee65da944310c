"""The device projection (values as a product over the terms, maps and filters
on the matrix cores) at every order against the oracle.

Term counts 1, 5 and 17 leave a step of four terms part empty and take a second
round of sixteen.  Bar: identical node sets and 1e-13 relative L2, as for the
other projections (a dozen separable passes of at most 20 terms, exponentials
rounded differently).
"""
import numpy as np
import pytest

from mrcpp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [3, 5, 7, 9])
def test_projection_of_every_order_and_term_count(mr, orc, order):
    mra, omra = mr.MultiResolutionAnalysis((-8, 8), order), orc.OracleMRA((-8, 8), order)
    prec = 10.0 ** -(order // 2 + 1)
    for terms in (1, 5, 17):
        src = W.random_sources(30 + terms, terms, center_range=2.0, beta_range=(1.0, 30.0))
        f, of = mr.FunctionTree(mra), orc.OracleTree(omra)
        gx = mr.GaussExp.from_sources(src)
        mr.set_projection_target("device")
        try:
            mr.build_grid(f, gx)
            mr.project(prec, f, gx)
        finally:
            mr.set_projection_target("auto")
        of.project_gaussians(prec, src.coefs, src.exponents, src.centers)
        (mi, mc, mn), (oi, oc, on) = f.export(), of.export()
        assert np.array_equal(mi, oi)
        assert np.linalg.norm(mc - oc) <= 1e-13 * np.linalg.norm(oc)
        assert np.allclose(mn, on, rtol=1e-12, atol=1e-12 * np.abs(on).max())
