"""Streamed downloads and the handing over of a tree's coefficients.

mwg_download_stream must deliver every byte once and in order for pieces at
the edges of its ring (one piece, as many as the ring holds, one more, a short
last one), and refuse a piece size outside its range.  A tree whose
coefficients live on the GPU must give the same arrays when exported again,
after its host copy is made (evalf) and when it has as many nodes as make
several pieces; the exported coefficients must match the norms beside them.
"""
import ctypes

import numpy as np
import pytest

from mrcpp_amd import workloads as W

pytestmark = pytest.mark.gpu

SINK = ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t)


@pytest.mark.parametrize("nbytes,piece", [(1, 4096), (4096, 4096), (4 * 4096, 4096), (5 * 4096, 4096), (37 * 4096 + 5, 4096), (9 << 20, 4 << 20)])
def test_stream_delivers_every_byte_in_order(mr, nbytes, piece):
    L = mr.lib()
    assert L.mwg_init(0) == 0
    L.mwg_download_stream.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_size_t, SINK, ctypes.c_void_p]
    a = np.random.default_rng(nbytes).integers(0, 256, nbytes).astype(np.uint8)
    p = ctypes.c_void_p()
    assert L.mwg_malloc(ctypes.byref(p), nbytes) == 0
    try:
        assert L.mwg_upload(p, a.ctypes.data, nbytes) == 0
        got = []
        sink = SINK(lambda ctx, q, off, n: got.append((off, ctypes.string_at(q, n))))
        assert L.mwg_download_stream(p, nbytes, piece, sink, None) == 0, L.mwg_last_error()
        assert [o for o, _ in got] == list(range(0, nbytes, piece))
        assert b"".join(b for _, b in got) == a.tobytes()
        for bad in (0, (4 << 20) + 1):
            assert L.mwg_download_stream(p, nbytes, bad, sink, None) != 0
    finally:
        L.mwg_free(p)


@pytest.mark.parametrize("order,prec,n", [(3, 1e-2, 1), (7, 1e-6, 16)])
def test_export_is_repeatable_and_whole(mr, order, prec, n):
    mra = mr.MultiResolutionAnalysis((-32, 32), order)
    f = mr.FunctionTree(mra)
    g = mr.GaussExp.from_sources(W.random_sources(20240607, n, 4.0))
    mr.build_grid(f, g)
    mr.project(prec, f, g)
    P = mr.PoissonOperator(mra, prec)
    v = mr.FunctionTree(mra)
    mr.apply(prec, v, P, f)
    for t in (f, v):
        i0, c0, n0 = t.export()
        i1, c1, n1 = t.export()
        e = t.evalf((0.1, 0.2, 0.3))  # makes the host copy
        i2, c2, n2 = t.export()
        assert t.evalf((0.1, 0.2, 0.3)) == e
        for i, c, m in ((i1, c1, n1), (i2, c2, n2)):
            assert np.array_equal(i0, i) and np.array_equal(c0, c) and np.array_equal(n0, m)
        # each row is its own node's: its square norm is beside it (a sum of 8 (k+1)^3 squares)
        sq = np.sum(c0 * c0, axis=1)
        assert np.all(np.abs(sq - n0[:, 8]) <= 1e-12 * np.maximum(sq, n0[:, 8]) + 1e-300)
        assert t.export(with_coefs=False)[1] is None
