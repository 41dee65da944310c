"""The one-wave-per-item band kernels at the edges of their work split.

Reference: the FP64 vector-ALU kernel (`fp64_vector`), which shares none of
their tiles, operand layouts or partial-slot order.  Cases: every order; units
of 8 groups (many slots per node), of 64 and 65 (the 64-record chunk and one
past it) and of 1024 (most nodes a single unit, written without a slot);
worlds of one and of several root boxes.  Both sum the same products in another
order: held to the FP64 bar of the parity tests, 1e-12.
"""
import sys

import numpy as np
import pytest

from mrcpp_amd import workloads as W

pytestmark = pytest.mark.gpu

CASES = [(3, 1e-3, None, (-16, 16)), (5, 1e-4, 1.2, (-20, 20)), (7, 1e-4, None, (-3, (0, -1, 0), (1, 2, 1))), (9, 1e-5, 0.7, (-20, 20))]


@pytest.fixture
def settings(mr):
    yield
    mr.set_band_launch(32, 0)
    mr.set_sweep_precision("fp64")


@pytest.mark.parametrize("order,prec,mu,box", CASES)
def test_waves_equal_vector_kernel(mr, settings, order, prec, mu, box):
    mra = mr.MultiResolutionAnalysis(box, order)
    src = W.random_sources(5, 2, 1.5)
    src.centers = [tuple(abs(x) for x in c) for c in src.centers]  # inside every world
    f = mr.FunctionTree(mra)
    g = mr.GaussExp.from_sources(src)
    mr.build_grid(f, g)
    mr.project(prec, f, g)
    P = mr.PoissonOperator(mra, prec) if mu is None else mr.HelmholtzOperator(mra, mu, prec)

    def apply(precision, unit_groups, per_cu=0):
        print("case order", order, precision, unit_groups, per_cu, file=sys.stderr, flush=True)
        mr.set_sweep_precision(precision)
        mr.set_band_launch(unit_groups, per_cu)
        out = mr.FunctionTree(mra)
        st = mr.apply(prec, out, P, f)
        return out.export(), int(st["n_applied"])

    (ri, rc, rn), rt = apply("fp64_vector", 32)
    for unit_groups, per_cu in ((8, 0), (64, 1), (65, 0), (1024, 0)):
        (i, c, n), t = apply("fp64", unit_groups, per_cu)
        assert np.array_equal(i, ri) and t == rt, (unit_groups, t, rt)
        assert np.linalg.norm(c - rc) <= 1e-12 * np.linalg.norm(rc), unit_groups
        assert np.linalg.norm(n - rn) <= 1e-12 * np.linalg.norm(rn), unit_groups
