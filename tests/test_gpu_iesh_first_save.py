"""EhrenfestNA: the first save follows the first acceleration directly, and both use the same LDS scratch.  Many copies
of a few initial states have to stay bitwise the same trajectory in every workgroup (mean-field dynamics draws no
numbers), and the trajectory is the oracle's."""
import numpy as np
import pytest

import test_gpu_iesh as T

pytestmark = pytest.mark.gpu


# two, three and seven wavefronts a trajectory, and a single one, which needs no barrier
@pytest.mark.parametrize("M,Ne,copies", [(15, 8, 2000), (17, 9, 2000), (40, 20, 2000), (100, 50, 200)])
def test_copies_stay_the_same(oracle, key, M, Ne, copies):
    from nqcd_mi355x import _lib as L
    r0, v0, occ0 = T._inputs(4, Ne, 5 + M)
    many = np.tile(r0, copies), np.tile(v0, copies), np.tile(occ0, (copies, 1))
    g = T._gpu(L, L.METHOD_EHRENFEST_NA, M, Ne, *many, 2.0, 3, key, save_every=1)
    for f in ("r", "v", "psi", "di", "ad"):
        a = g[f].reshape((copies, 4) + g[f].shape[1:])
        assert (a == a[:1]).all(), f
    c = T._cpu(oracle, 1, M, Ne, r0, v0, occ0, 2.0, 3, key, save_every=1)
    T._compare({k: g[k][:4] for k in ("r", "v", "psi", "di")}, c, hops=False)
