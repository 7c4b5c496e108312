"""The spin-boson kernel with FP32 nuclei: the rounding of its bath against a plain FP32 velocity Verlet, and hops,
rescaling and ragged ensemble sizes against the oracle."""
import numpy as np
import pytest

from test_gpu_spin_boson import N, _debye, _wigner

pytestmark = pytest.mark.gpu
F32 = np.float32


def _fma(a, b, c):
    return F32(np.float64(a) * np.float64(b) + np.float64(c))


def test_bath_rounding(oracle, key):
    """Without coupling between the states the bath is N oscillators under a constant force.  The kernel's rounding
    error over 1000 steps must not pass that of velocity Verlet step by step in FP32 (every half kick formed first and
    subtracted once), both measured against the same steps in FP64 from the same FP32 coefficients and positions.  The
    kernel rounds a velocity once a step where that form does twice, so the bound is the form's own error."""
    from nqcd_mi355x import _lib as L
    w, c = _debye(oracle)
    sdr, sdv = _wigner(w, 5.0)
    dt, ntraj, nsteps = 0.002, 400, 1000
    out = []
    for n in (0, nsteps):
        E = L.Ensemble(0)
        E.set_problem(1, 2, 1, N, np.ones(N), dt, precision=L.PREC_FP32_NUCLEI)
        E.set_model(0, L.MODEL_SPIN_BOSON, np.concatenate([[1e3, 0.0], w, c]))   # lower state: force -c
        E.sample_initial(L.SAMPLER_HARMONIC_WIGNER, ntraj, np.concatenate([np.zeros(N), sdr, np.zeros(N), sdv]), key,
                         initial_state=0, state_basis=0)
        E.run(0.0, n * dt, key)
        out += [E.download(L.FIELD_R).reshape(ntraj, N), E.download(L.FIELD_V).reshape(ntraj, N)]
        E.close()
    x0, v0, xg, vg = out
    assert np.array_equal(x0, F32(x0)) and np.array_equal(v0, F32(v0))
    kx, kf, d = F32(0.5 * dt * w * w), F32(0.5 * dt * c), F32(dt)
    x, v = x0.copy(), v0.copy()
    xs, vs = F32(x0), F32(v0)
    for _ in range(nsteps):
        v = v - (kx.astype(float) * x - kf)
        x = x + float(d) * v
        v = v - (kx.astype(float) * x - kf)
        vs = vs - _fma(kx, xs, -kf)
        xs = _fma(d, vs, xs)
        vs = vs - _fma(kx, xs, -kf)
    for got, plain, ref in ((xg, xs, x), (vg, vs, v)):
        err, bound = np.sqrt(((got - ref) ** 2).mean()), np.sqrt(((plain - ref) ** 2).mean())
        print(f"rms error {err:.3g}, plain form {bound:.3g}")
        assert err <= bound
