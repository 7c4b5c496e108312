"""Per-trajectory results on the host: runs of zero steps give back what was loaded, in its place, at the edges
of the 64 x 16 tiles of the transposition and over more than one chunk of its staging buffer."""
import numpy as np
import pytest

import nstate_models as NS

pytestmark = pytest.mark.gpu


def _beads(L, P, r, v):
    E = L.Ensemble(0)
    E.set_problem(L.METHOD_RPMD, 1, 1, 1, [1836.0], 1.0, algorithm=L.ALG_BCB, nbeads=P, temperature=0.1)
    E.set_model(0, L.MODEL_DW_GAUSSIAN, [1 / 1200, 1 / 40, 0.0, 0.0, 1.0])
    E.load_initial(r, v, None)
    E.run(0.0, 0.0, 1)
    out = E.download(L.FIELD_R), E.download(L.FIELD_V)
    E.close()
    return out


# 300001 x 32 beads: 77 MB, two chunks of the 64 MB staging buffer
@pytest.mark.parametrize("P,ntraj", [(1, 65), (2, 1), (4, 63), (16, 64), (32, 65), (64, 127), (32, 300001)])
def test_rows(P, ntraj):
    from nqcd_mi355x import _lib as L
    r = np.arange(ntraj * P, dtype=float).reshape(ntraj, P) / 1024.0
    v = -r / 3.0
    gr, gv = _beads(L, P, r, v)
    # to normal modes and back: two orthogonal P x P products, each within P roundings of the row's norm
    # (at most 8e-10, where neighbours differ by 1e-3 and 3e-4)
    tol = 4 * P * 2.0 ** -53 * np.linalg.norm(r, axis=1, keepdims=True)
    assert (np.abs(gr.reshape(ntraj, P) - r) <= tol).all()
    assert (np.abs(gv.reshape(ntraj, P) - v) <= tol).all()


@pytest.mark.parametrize("n", [2, 3, 5, 8])
@pytest.mark.parametrize("ntraj", [1, 64, 129])
def test_density(n, ntraj):
    """The n-state densities, whose imaginary parts lie behind the real ones."""
    from nqcd_mi355x import _lib as L
    rng = np.random.default_rng(n)
    s = rng.normal(size=(ntraj, n, n)) + 1j * rng.normal(size=(ntraj, n, n))
    s = s + s.conj().transpose(0, 2, 1)
    E = L.Ensemble(0)
    E.set_problem(L.METHOD_EHRENFEST, n, 1, 1, [NS.MASS], 1.0)
    E.set_model(0, L.MODEL_MORSE_N, [n] + NS.morse_table(n))
    E.load_initial(np.full((ntraj, 1), 3.2), np.zeros((ntraj, 1)), s)
    E.run(0.0, 0.0, 1)
    g = E.download(L.FIELD_SIGMA_RE) + 1j * E.download(L.FIELD_SIGMA_IM)
    E.close()
    assert np.array_equal(g, s)
