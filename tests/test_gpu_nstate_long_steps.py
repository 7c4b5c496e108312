"""Three long FP32 steps of the n-state density, the first from the zero buffers of the run's start: there the generator
grows from nothing to a norm of 5 to 450 (about 8, the limit of one part for such a step, and 12, the limit for a steady
one, among them), so that the parts which the step is cut into and their orders have to be as many as its end asks for.
Against the oracle's sub-steps, 4000 of them (a norm of 0.1 each at most, their error below 1e-8)."""
import numpy as np
import pytest

import nstate_models as NS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,dt", [(3, 500.0), (3, 1200.0), (4, 1500.0), (4, 3000.0), (8, 300.0), (8, 700.0),
                                  (3, 60.0), (3, 100.0), (3, 104.0), (3, 150.0), (3, 6000.0), (8, 3000.0)])
def test_long_steps(oracle, n, dt):
    from nqcd_mi355x import _lib as L
    mass, ntraj = 1e9, 65   # heavy: the position changes by 0.1 bohr at most
    table = NS.three_state() if n == 3 else NS.morse_table(n)
    rng = np.random.default_rng(n)
    r0, v0 = rng.normal(3.2, 0.02, (ntraj, 1)), np.full((ntraj, 1), 0.02 / dt)
    r0, v0 = np.float32(r0).astype(float), np.float32(v0).astype(float)
    c = rng.normal(size=(ntraj, n)) + 1j * rng.normal(size=(ntraj, n))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    sig0 = c[:, :, None] * c[:, None, :].conj()
    E = L.Ensemble(0)
    E.set_problem(L.METHOD_EHRENFEST, n, 1, 1, [mass], dt, precision=L.PREC_FP32_NUCLEI)
    E.set_model(0, L.MODEL_MORSE_N, [n] + table)
    E.load_initial(r0, v0, sig0)
    E.run(0.0, 3 * dt, 1)
    s = E.download(L.FIELD_SIGMA_RE) + 1j * E.download(L.FIELD_SIGMA_IM)
    E.close()
    o = oracle.run_ensemble(1, oracle.make_model(oracle.MODEL_MORSE_N, n, 1, table), mass, r0, v0, sig0, dt=dt, nsteps=3, key=1,
                            nsub=4000)
    # the phase of 3 dt x (energies of at most 0.5 within four FP32 roundings, and a slope of at most 0.5 times the
    # rounding of a position of 3.2)
    tol = 3 * dt * (4 * 0.5 * 6e-8 + 0.5 * 2.4e-7)
    assert np.abs(s - (o["sig_re"] + 1j * o["sig_im"])).max() < tol
