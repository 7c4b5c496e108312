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


@pytest.mark.parametrize("coupling", [0.0, 1e-150, 3e-141, 1e-12, 0.005, 0.3])
def test_two_state_eigenvectors(oracle, coupling):
    """From exactly degenerate diabats to strong coupling: splittings whose square leaves the range of a double take
    the square roots themselves.  Two steps from rest at and around the crossing, so that every lane keeps its splitting.
    FP64 coordinates only: in FP32 the model itself is degenerate within 1e-8 of the crossing."""
    from nqcd_mi355x import _lib as L
    p = [0.01, 1.6, coupling, 1.0]
    r0 = np.array([0.0, 0.0, 1e-15, -1e-9, 1e-3, -0.4, 2.0, -3.0])[:, None]
    sig0 = np.zeros((8, 2, 2), complex)
    sig0[:, 0, 0], sig0[:, 1, 1] = 0.75, 0.25
    E = L.Ensemble(0)
    E.set_problem(L.METHOD_EHRENFEST, 2, 1, 1, [MASS], 0.1)
    E.set_model(0, 0, p)
    E.load_initial(r0, np.zeros((8, 1)), sig0)
    E.run(0.0, 0.2, 1)
    r, v = E.download(L.FIELD_R), E.download(L.FIELD_V)
    E.close()
    c = oracle.run_ensemble(1, oracle.make_model(0, 2, 1, p), MASS, r0, np.zeros((8, 1)), sig0, dt=0.1, nsteps=2, key=1)
    # a coupling of 1e-150 at the crossing itself: the derivative coupling's square overflows, here and there alike
    bad = np.isnan(c["v"])
    assert np.array_equal(np.isnan(v), bad) and np.array_equal(np.isnan(r), np.isnan(c["r"]))
    assert coupling in (0.0, 1e-150, 3e-141) or not bad.any()
    # accelerations of at most 0.016 / 2000 over 0.2, velocities of 1.6e-6, to 1e-12 of that: a dozen roundings make 3e-15
    assert np.nanmax(np.abs(v - c["v"])) < 1.6e-18
    assert np.nanmax(np.abs(r - c["r"])) < 1e-15   # positions of 3 rounded twice
