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


@pytest.mark.parametrize("ntraj", [1, 65, 513])
@pytest.mark.parametrize("rescaling", [0, 1, 2])
def test_fssh(oracle, key, ntraj, rescaling):
    """Hops, frustrated hops and their velocity changes, with bath masses that differ.  Velocities a tenth of the
    thermal ones, so that part of the hops upwards lack the energy."""
    from nqcd_mi355x import _lib as L
    w, c = _debye(oracle)
    sdr, sdv = _wigner(w, 5.0)
    sdv = 0.1 * sdv
    mass = 1.0 + 0.5 * np.cos(np.arange(N))
    dt, nsteps = 0.002, 60
    E = L.Ensemble(0)
    E.set_problem(0, 2, 1, N, mass, dt, rescaling=rescaling, precision=L.PREC_FP32_NUCLEI)
    E.set_model(0, L.MODEL_SPIN_BOSON, np.concatenate([[1.0, 1.0], w, c]))
    E.sample_initial(L.SAMPLER_HARMONIC_WIGNER, ntraj, np.concatenate([np.zeros(N), sdr, np.zeros(N), sdv]), key,
                     initial_state=1, state_basis=0)
    E.run(0.0, nsteps * dt, key, save_every=1)
    g = {"r": E.download(L.FIELD_R), "v": E.download(L.FIELD_V), "pop_di": E.download(L.FIELD_SAVE_POP_DI)}
    states, nhops = E.download(L.FIELD_SAVE_STATE), E.download(L.FIELD_NHOPS)
    E.close()

    m = oracle.make_model(oracle.MODEL_SPIN_BOSON, 2, N, [1.0, 1.0], omega=w, cbath=c)
    r0, v0 = oracle.sample_gaussian(ntraj, N, 0.0, sdr[None, :], 0.0, sdv[None, :], key)
    sig0 = np.zeros((ntraj, 2, 2), complex)
    sig0[:, 1, 1] = 1.0

    def cpu(r, v, resc):
        return oracle.run_ensemble(0, m, mass, r, v, sig0, state0=np.ones(ntraj, np.int32), dt=dt, nsteps=nsteps,
                                   save_every=1, nsave=nsteps + 1, key=key, rescaling=resc)

    o, p = cpu(r0, v0, rescaling), cpu(F32(r0).astype(float), F32(v0).astype(float), rescaling)
    same = (states == o["save_state"]).all(axis=1) & (nhops == o["nhops"])
    # a rounding of 6e-8 moves one of ntraj x 60 decisions with a probability of the same order
    assert (~same).sum() <= ntraj // 100
    # a step rounds positions and velocities once each, and its coefficients and time step: each does at most what the
    # rounding of the initial positions and velocities does (p against o)
    for f in ("r", "v", "pop_di"):
        size = np.abs(p[f] - o[f])[(p["save_state"] == o["save_state"]).all(axis=1)].max()
        assert np.abs(g[f].reshape(o[f].shape) - o[f])[same].max() <= (4 * nsteps + 1) * max(size, 6e-8), f
    if ntraj == 513:
        assert o["nhops"].sum() > 1000
        if rescaling < 2:   # reflected, or not, on some trajectories
            assert (np.abs(o["v"] - cpu(r0, v0, 1 - rescaling)["v"]).reshape(ntraj, -1).max(axis=1) > 0).sum() > 20
