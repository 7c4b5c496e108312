"""Few trajectories with many saves on the host: values against the device's reductions and against runs of one
trajectory, over more rows than one pass of the transposition's grid, and a time of the order of a plain copy."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MASS = 2000.0


def _ensemble(L, r0, nsteps, key, save_every=1):
    n = len(r0)
    sig = np.zeros((n, 2, 2), complex)
    sig[:, 0, 0] = 1.0
    E = L.Ensemble(0)
    E.set_problem(L.METHOD_EHRENFEST, 2, 1, 1, [MASS], 1.0)
    E.set_model(0, L.MODEL_TULLY1, [0.01, 1.6, 0.005, 1.0])
    E.load_initial(r0[:, None], np.full((n, 1), 15.0 / MASS), sig)
    E.run(0.0, float(nsteps), key, save_every=save_every)
    return E


# 65 trajectories of 20001 saves: 2501 tiles of rows on a grid of 2048
@pytest.mark.parametrize("ntraj,nsteps", [(1, 7), (1, 5000), (2, 3001), (65, 20000)])
def test_values(key, ntraj, nsteps):
    from nqcd_mi355x import _lib as L
    r0 = np.linspace(-5.0, -3.0, ntraj)
    E = _ensemble(L, r0, nsteps, key)
    pop, kin = E.download(L.FIELD_SAVE_POP_AD), E.download(L.FIELD_SAVE_EKIN)
    mean = E.reduce(L.OUT_ADIABATIC_POPULATION, L.RED_MEAN, 2 * E.nsave)
    E.close()
    pop, kin = pop.reshape(ntraj, nsteps + 1, 2), kin.reshape(ntraj, nsteps + 1)
    assert np.abs(pop.mean(axis=0).ravel() - mean).max() < 1e-13   # sums of ntraj numbers below one
    for i in sorted({0, ntraj // 2, ntraj - 1}):
        S = _ensemble(L, r0[i:i + 1], nsteps, key)
        assert np.array_equal(S.download(L.FIELD_SAVE_POP_AD).reshape(nsteps + 1, 2), pop[i])
        assert np.array_equal(S.download(L.FIELD_SAVE_EKIN).reshape(nsteps + 1), kin[i])
        S.close()


@pytest.mark.parametrize("ntraj", [1, 2])
def test_time(key, ntraj):
    """The populations of 1e5 saves take no more than eight times as long as as many numbers that are one row on the
    device already (with one workgroup for all rows they took sixty to ninety times as long)."""
    from nqcd_mi355x import _lib as L

    def best(E, field):
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            E.download(field)
            t.append(time.perf_counter() - t0)
        return min(t)

    E = _ensemble(L, np.full(ntraj, -5.0), 100_000, key)
    tall = best(E, L.FIELD_SAVE_POP_AD)
    E.close()
    E = _ensemble(L, np.full(200_000 * ntraj, -5.0), 1, key, save_every=0)
    flat = best(E, L.FIELD_SAVE_EKIN)
    E.close()
    print(f"{ntraj} trajectories: {1e3 * tall:.3f} ms against {1e3 * flat:.3f} ms")
    assert tall < 8 * flat
