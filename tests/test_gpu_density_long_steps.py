"""Two-state launches of long steps, on both sides of the limits beyond which a launch takes the sub-steps throughout
(gap x dt = 0.45 with FP64 nuclei, 1.9 with FP32): results against the oracle, and a time that is that of the sub-steps
and not of both forms together."""
import numpy as np
import pytest

from test_gpu_density_series import MASS, TULLY, _inputs, _run

pytestmark = pytest.mark.gpu
GAP = {0: 2 * np.hypot(0.01, 0.005), 1: np.hypot(0.05, 0.03), 2: 2 * np.hypot(6e-4, 0.2)}


@pytest.mark.parametrize("kind", [0, 1, 2])
@pytest.mark.parametrize("precision,z", [(0, 0.44), (0, 0.46), (0, 3.0), (1, 1.88), (1, 1.92)])
def test_values(oracle, kind, precision, z):
    dt, n, nsteps = z / GAP[kind], 193, 12
    r0, v0, sig0 = _inputs(n)
    v0 = v0 / max(1.0, dt / 4.0)   # as far a step as at dt = 4
    m = oracle.make_model(kind, 2, 1, TULLY[kind])
    c = oracle.run_ensemble(1, m, MASS, r0, v0, sig0, dt=dt, nsteps=nsteps, key=1)
    r, v, s = _run(kind, dt, nsteps, r0, v0, sig0, precision, 5)
    err = np.abs(s - (c["sig_re"] + 1j * c["sig_im"])).max()
    if precision == 0:
        assert err < 1e-10 and np.allclose(r, c["r"], rtol=1e-10, atol=1e-10)
    else:
        # FP32 positions of 4 bohr, 12 roundings through gradients of at most 0.1 and 12 dt of phase, and the sub-steps'
        # own error of at most 1e-5 a step, which the series has to its last orders only
        assert err < 12 * 4 * 6e-8 * 0.1 * 12 * dt + 12e-5


@pytest.mark.parametrize("kind,precision,z", [(0, 0, 0.65), (1, 0, 0.65), (1, 1, 2.5), (2, 1, 4.5)])
def test_time(key, kind, precision, z):
    """Five sub-steps take no longer than the mean of four and six, which never take the series (with both forms in most
    wavefronts they took 1.12 to 1.2 times as long)."""
    from nqcd_mi355x import _lib as L
    dt, n = z / GAP[kind], 200_000
    rng = np.random.default_rng(1)
    r0, v0 = rng.normal(-5, 0.7, (n, 1)), rng.uniform(10, 30, (n, 1)) / MASS
    sig0 = np.zeros((n, 2, 2), complex)
    sig0[:, 0, 0] = 1.0
    t = {}
    for nsub in (4, 5, 6):
        E = L.Ensemble(0)
        E.set_problem(L.METHOD_FSSH, 2, 1, 1, [MASS], dt, precision=precision, electronic_substeps=nsub)
        E.set_model(0, kind, TULLY[kind])
        E.load_initial(r0, v0, sig0, state=np.zeros(n, np.int32))
        t[nsub] = min(E.run(0.0, 60 * dt, key)["kernel_ms"] for _ in range(6))
        E.close()
    print(t)
    assert t[5] < 1.06 * 0.5 * (t[4] + t[6])
