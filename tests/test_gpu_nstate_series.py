"""The n-state density's power series: every state count, the limits of its orders and the parts a long FP32 step is
cut into, and the kernels of other sub-step counts, against the oracle.  The generator of the Morse chains has a norm
of about 0.05 dt, so dt = 0.5 ... 80 passes every limit (z2 = 0.0041 ... 4) and reaches several parts."""
import numpy as np
import pytest

import nstate_models as NS

pytestmark = pytest.mark.gpu


def _run(n, table, dt, nsteps, precision, nsub, r0, v0, sig0):
    from nqcd_mi355x import _lib as L
    E = L.Ensemble(0)
    E.set_problem(1, n, 1, 1, [NS.MASS], dt, precision=precision, electronic_substeps=nsub)
    E.set_model(0, L.MODEL_MORSE_N, [n] + table)
    E.load_initial(r0, v0, sig0)
    E.run(0.0, nsteps * dt, 1)
    out = E.download(L.FIELD_R), E.download(L.FIELD_SIGMA_RE) + 1j * E.download(L.FIELD_SIGMA_IM)
    E.close()
    return out


def _inputs(n, ntraj):
    rng = np.random.default_rng(n)
    r0 = rng.normal(3.2, 0.2, (ntraj, 1))
    v0 = np.sqrt(2 * rng.uniform(0.02, 0.04, (ntraj, 1)) / NS.MASS)
    c = rng.normal(size=(ntraj, n)) + 1j * rng.normal(size=(ntraj, n))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    return r0, v0, c[:, :, None] * c[:, None, :].conj()


def _oracle(oracle, n, table, dt, nsteps, nsub, r0, v0, sig0):
    m = oracle.make_model(oracle.MODEL_MORSE_N, n, 1, table)
    c = oracle.run_ensemble(1, m, NS.MASS, r0, v0, sig0, dt=dt, nsteps=nsteps, key=1, nsub=nsub)
    return c["r"], c["sig_re"] + 1j * c["sig_im"]


@pytest.mark.parametrize("n", [2, 3, 4, 5, 8])
@pytest.mark.parametrize("dt", [0.5, 2.0, 6.0, 20.0, 80.0])
def test_series(oracle, n, dt):
    table = NS.three_state() if n == 3 else NS.morse_table(n)
    ntraj, nsteps = 67, 20
    r0, v0, sig0 = _inputs(n, ntraj)
    # FP64: the sub-steps' result (1e-12 a step by the rule; the window tolerance of the parity tests)
    r, s = _run(n, table, dt, nsteps, 0, 5, r0, v0, sig0)
    ro, so = _oracle(oracle, n, table, dt, nsteps, 5, r0, v0, sig0)
    assert np.allclose(r, ro, rtol=1e-9, atol=1e-10)
    assert np.abs(s - so).max() < 1e-9
    # FP32: the equation's solution (an oracle of 400 sub-steps); 20 roundings of 4 bohr by 2^-24 through energy
    # differences whose slope is at most 0.05 over 20 dt of phase, and the force's response to them
    r, s = _run(n, table, dt, nsteps, 1, 5, r0, v0, sig0)
    ro, so = _oracle(oracle, n, table, dt, nsteps, 400, r0, v0, sig0)
    tol = 20 * 4 * 6e-8 * 0.05 * 20 * dt + 1e-5
    assert np.abs(s - so).max() < tol
    assert np.abs(r - ro).max() < 1e-4


@pytest.mark.parametrize("nsub", [1, 4, 7])
def test_other_sub_step_counts(oracle, nsub):
    n, dt, nsteps = 3, 4.0, 20
    table = NS.three_state()
    r0, v0, sig0 = _inputs(n, 67)
    r, s = _run(n, table, dt, nsteps, 0, nsub, r0, v0, sig0)
    ro, so = _oracle(oracle, n, table, dt, nsteps, nsub, r0, v0, sig0)
    assert np.allclose(r, ro, rtol=1e-9, atol=1e-10) and np.abs(s - so).max() < 1e-9
