"""The wave kernels of the band sum need no more device memory than the
tile-shared kernel on the same levels (order 7 runs both).

Scratch grows on demand and is kept, so a fresh process applies a batch with
the tile layout, then with the wave kernels, and compares the free device
memory.  Allowed: the wave kernels' unit records, 48 bytes a unit where the
tile kernel has 16, for 2^30 / 2^15 slots and the nodes of a level (no more than
the trees have), a quarter more by the growth rule.
"""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import torch
import mrcpp_amd as mr
from mrcpp_amd import workloads as W

mra = mr.MultiResolutionAnalysis((-32, 32), 7)
tasks = []
for b in W.batch_sources()[:8]:
    f = mr.FunctionTree(mra)
    gx = mr.GaussExp.from_sources(b["sources"])
    mr.build_grid(f, gx)
    mr.project(b["prec"], f, gx)
    tasks.append((b["prec"], mr.PoissonOperator(mra, b["prec"]) if b["mu"] is None else mr.HelmholtzOperator(mra, b["mu"], b["prec"]), f))


def free_after(layout):
    mr.set_band_layout(layout)
    for _ in range(2):
        outs = [mr.FunctionTree(mra) for _ in tasks]
        stats = mr.apply_batch([(p, o, P, f) for (p, P, f), o in zip(tasks, outs)])
        mr.device_synchronize()
        del outs
    return torch.cuda.mem_get_info()[0], sum(int(s["n_output_nodes"]) for s in stats)


(tiles, nodes), (rows, _) = free_after("tiles"), free_after("rows")
print(tiles - rows, nodes)
"""


def test_wave_kernels_need_no_more_scratch(mr):
    r = subprocess.run([sys.executable, "-c", CHILD], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    grown, nodes = map(int, r.stdout.split()[-2:])
    print("grown by", grown, "trees of", nodes, "nodes")
    assert grown <= (2 ** 15 + nodes) * 32 * 5 // 4
