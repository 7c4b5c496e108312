"""The density's power series over a nuclear step (series_step2 of nqcd_device.h) against the oracle's five Tsit5
sub-steps.  Time steps from 0.05 to 10 a.u. take the accumulated norm of the generator across every limit of the
series' orders (z2 = 0.0041 ... 0.99, FP32: 4) and past the last one, where the sub-steps are taken themselves.
Per step the two differ by at most 1e-12 in FP64 (the rule's own limit); 40 steps of Ehrenfest dynamics, whose
forces read the density, keep that within 1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MASS = 2000.0
TULLY = {0: [0.01, 1.6, 0.005, 1.0], 1: [0.1, 0.28, 0.015, 0.06, 0.05], 2: [6e-4, 0.1, 0.9]}


def _inputs(n):
    rng = np.random.default_rng(8)
    r0 = rng.uniform(-4.0, 4.0, (n, 1))
    v0 = rng.uniform(-30.0, 30.0, (n, 1)) / MASS
    c = rng.normal(size=(n, 2)) + 1j * rng.normal(size=(n, 2))
    c /= np.linalg.norm(c, axis=1, keepdims=True)
    return r0, v0, c[:, :, None] * c[:, None, :].conj()   # pure states with every component of the density


def _run(kind, dt, nsteps, r0, v0, sig0, precision, nsub):
    from nqcd_mi355x import _lib as L
    E = L.Ensemble(0)
    E.set_problem(L.METHOD_EHRENFEST, 2, 1, 1, [MASS], dt, precision=precision, electronic_substeps=nsub)
    E.set_model(0, kind, TULLY[kind])
    E.load_initial(r0, v0, sig0)
    E.run(0.0, nsteps * dt, 1)
    out = E.download(L.FIELD_R), E.download(L.FIELD_V), \
        E.download(L.FIELD_SIGMA_RE) + 1j * E.download(L.FIELD_SIGMA_IM)
    E.close()
    return out


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("dt", [0.05, 0.4, 1.0, 2.5, 4.0, 10.0])
def test_series_against_sub_steps(oracle, kind, dt):
    n, nsteps = 193, 40
    r0, v0, sig0 = _inputs(n)
    m = oracle.make_model(kind, 2, 1, TULLY[kind])
    c = oracle.run_ensemble(1, m, MASS, r0, v0, sig0, dt=dt, nsteps=nsteps, key=1)
    sc = c["sig_re"] + 1j * c["sig_im"]
    r, v, s = _run(kind, dt, nsteps, r0, v0, sig0, 0, 5)
    assert np.abs(s - sc).max() < 1e-10
    assert np.allclose(r, c["r"], rtol=1e-10, atol=1e-10) and np.allclose(v, c["v"], rtol=1e-9, atol=1e-12)
    if dt <= 4.0:
        # FP32 coordinates: 40 roundings of 6e-8 on positions of up to 4 bohr, through gradients of at most 0.1 and
        # 40 dt of phase: 40 * 4 * 6e-8 * 0.1 * 40 * dt = 4e-5 dt on the density
        _, _, s32 = _run(kind, dt, nsteps, r0, v0, sig0, 1, 5)
        assert np.abs(s32 - sc).max() < 4e-5 * dt + 1e-5


@pytest.mark.parametrize("nsub", [1, 4, 6])
def test_other_sub_step_counts_keep_tsit5(nsub):
    """Other counts than five run the sub-steps: their error at 1 sub-step is visible, and falls as theirs does."""
    r0, v0, sig0 = _inputs(64)
    ref = _run(2, 4.0, 10, r0, v0, sig0, 0, 40)[2]
    err = np.abs(_run(2, 4.0, 10, r0, v0, sig0, 0, nsub)[2] - ref).max()
    lo, hi = {1: (1e-5, 1e-1), 4: (1e-9, 1e-5), 6: (1e-10, 1e-6)}[nsub]
    assert lo < err < hi
