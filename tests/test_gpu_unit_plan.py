"""The plan of a short level in one workgroup against the plan by scans.

A tree whose levels stay below 1024 nodes is applied alone (one workgroup) and
together with 23 others, whose joint levels exceed the bound (scans).  Units
depend on the node alone, so the results, norms and counts have to be the same
bits.  Order 3 also takes its partial sums and norms in one kernel, the other orders
in two.
"""
import numpy as np
import pytest

from mrcpp_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order,prec", [(3, 1e-3), (5, 1e-4)])
def test_short_and_long_levels_have_one_plan(mr, order, prec):
    mra = mr.MultiResolutionAnalysis((-16, 16), order)
    P = mr.PoissonOperator(mra, prec)
    trees = []
    for i in range(24):
        src = W.random_sources(60 + i, 2 + i % 3, center_range=4.0, beta_range=(1.0, 100.0))
        f = mr.FunctionTree(mra)
        gx = mr.GaussExp.from_sources(src)
        mr.build_grid(f, gx)
        mr.project(prec, f, gx)
        trees.append(f)
    alone, levels = [], []
    for f in trees:
        g = mr.FunctionTree(mra)
        st = mr.apply(prec, g, P, f)
        levels.append(st["level_nodes"])
        alone.append((g.export(), st["n_applied"]))
    joint = [sum(lv[d] for lv in levels if d < len(lv)) for d in range(max(map(len, levels)))]
    print(order, "widest level alone", max(map(max, levels)), "joint", max(joint))
    assert max(map(max, levels)) < 1024 < max(joint)
    outs = [mr.FunctionTree(mra) for _ in trees]
    stats = mr.apply_batch([(prec, o, P, f) for o, f in zip(outs, trees)])
    for (a, applied), o, st in zip(alone, outs, stats):
        b = o.export()
        assert all(np.array_equal(x, y) for x, y in zip(a, b))
        assert st["n_applied"] == applied
