"""IESH and EhrenfestNA kernels at the edges of their tiles: state counts on both sides of 16 and 32 (padding of the
rows and of the last products' steps), electron counts that leave half a column tile or fill the states (the kernels of
more column than row tiles), one electron, and the inverse of S for one to all columns of a wavefront.  Every step is
saved, so the populations' product runs beside every propagation."""
import numpy as np
import pytest

import test_gpu_iesh as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,Ne", [(15, 8), (15, 15), (16, 1), (17, 3), (30, 17), (31, 31), (32, 16), (47, 25), (79, 33), (95, 48),
                                  (111, 9)])
@pytest.mark.parametrize("method", [0, 1])
def test_edges(oracle, key, M, Ne, method):
    from nqcd_mi355x import _lib as L
    ntraj, nsteps = 5, 40
    r0, v0, occ0 = T._inputs(ntraj, Ne, 3 + M)
    g = T._gpu(L, L.METHOD_IESH if method == 0 else L.METHOD_EHRENFEST_NA, M, Ne, r0, v0, occ0, 2.0, nsteps, key, save_every=1)
    c = T._cpu(oracle, method, M, Ne, r0, v0, occ0, 2.0, nsteps, key, save_every=1)
    T._compare(g, c, hops=method == 0)
    assert np.allclose(g["di"].sum(axis=2), Ne, atol=1e-9)
