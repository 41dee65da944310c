"""Top-down reconstruction adds the two contributions of a direction to a child
one after the other, as the reference's accumulating filter passes do.

Filters with a one for every pair of children and the identity over the basis
hand a parent's blocks 0 and 4 to every child exactly, so each child has to be
(old + block 0) + block 4 to the last bit.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kp1", [4, 6, 8, 10])
def test_contributions_are_added_in_turn(mr, kp1):
    L = mr.lib()
    assert L.mwg_init(0) == 0
    n3, parents = kp1 ** 3, 3
    stride = 8 * n3
    rng = np.random.default_rng(kp1)
    coef = np.zeros((parents + 8 * parents, stride))
    coef[:parents, :n3] = rng.standard_normal((parents, n3))
    coef[:parents, 4 * n3:5 * n3] = rng.standard_normal((parents, n3))
    coef[parents:] = rng.standard_normal((8 * parents, stride))
    want = coef.copy()
    for k in range(parents):
        for c in range(8):
            child = want[parents + 8 * k + c]
            child[:n3] = (child[:n3] + coef[k, :n3]) + coef[k, 4 * n3:5 * n3]
    filters = np.tile(np.eye(kp1), (8, 1, 1))
    poff = stride * np.arange(parents, dtype=np.int64)
    coff = stride * (parents + 8 * np.arange(parents, dtype=np.int64))

    bufs = []

    def up(a):
        p = ctypes.c_void_p()
        assert L.mwg_malloc(ctypes.byref(p), a.nbytes) == 0
        bufs.append(p)
        assert L.mwg_upload(p, a.ctypes.data, a.nbytes) == 0
        return p

    try:
        d = [up(np.ascontiguousarray(a)) for a in (filters, coef, poff, coff)]
        L.mwg_reconstruct_add.argtypes = [ctypes.c_int] + [ctypes.c_void_p] * 4 + [ctypes.c_int, ctypes.c_longlong]
        assert L.mwg_reconstruct_add(kp1, d[0], d[1], d[2], d[3], parents, stride) == 0
        got = np.empty_like(coef)
        assert L.mwg_download(got.ctypes.data, d[1], got.nbytes) == 0
    finally:
        for p in bufs:
            L.mwg_free(p)
    assert np.array_equal(got, want)
