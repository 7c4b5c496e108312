"""The spin-boson kernel at ragged ensemble sizes (one lane, one past a wavefront), zero, one and a few steps, every
rescaling mode and bath masses that differ: positions partly in LDS, the two half kicks of a step end applied together
and the velocities' change of a hop as one pass of the wavefront, against the oracle."""
import numpy as np
import pytest

from test_gpu_spin_boson import N, _debye, _wigner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ntraj,nsteps", [(1, 60), (65, 60), (65, 1), (64, 0)])
@pytest.mark.parametrize("method,rescaling", [(0, 0), (0, 1), (0, 2), (1, 0)])
def test_ragged(oracle, key, ntraj, nsteps, method, rescaling):
    from nqcd_mi355x import _lib as L
    w, c = _debye(oracle)
    mass = 1.0 + 0.5 * np.cos(np.arange(N))
    sdr, sdv = _wigner(w, 5.0)
    dt = 0.002
    E = L.Ensemble(0)
    E.set_problem(method, 2, 1, N, mass, dt, rescaling=rescaling)
    E.set_model(0, L.MODEL_SPIN_BOSON, np.concatenate([[1.0, 1.0], w, c]))
    E.sample_initial(L.SAMPLER_HARMONIC_WIGNER, ntraj, np.concatenate([np.zeros(N), sdr, np.zeros(N), sdv]), key,
                     initial_state=1, state_basis=0)
    E.run(0.0, nsteps * dt, key, save_every=1)
    m = oracle.make_model(oracle.MODEL_SPIN_BOSON, 2, N, [1.0, 1.0], omega=w, cbath=c)
    r0, v0 = oracle.sample_gaussian(ntraj, N, 0.0, sdr[None, :], 0.0, sdv[None, :], key)
    sig0 = np.zeros((ntraj, 2, 2), complex)
    sig0[:, 1, 1] = 1.0
    o = oracle.run_ensemble(method, m, mass, r0, v0, sig0, state0=np.ones(ntraj, np.int32), dt=dt, nsteps=nsteps,
                            save_every=1, nsave=nsteps + 1, key=key, rescaling=rescaling)
    if method == 0:
        assert np.array_equal(E.download(L.FIELD_SAVE_STATE), o["save_state"])
        assert np.array_equal(E.download(L.FIELD_NHOPS), o["nhops"])
    # the window tolerance of the parity tests
    assert np.allclose(E.download(L.FIELD_R), o["r"], rtol=1e-9, atol=1e-11)
    assert np.allclose(E.download(L.FIELD_V), o["v"], rtol=1e-9, atol=1e-11)
    assert np.allclose(E.download(L.FIELD_SAVE_POP_DI), o["pop_di"], rtol=1e-9, atol=1e-11)
    E.close()
