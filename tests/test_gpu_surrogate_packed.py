"""The packed copy of the weights that the optimiser writes during training is the one that loading the same weights
makes: values, input gradients (which alone read some of its blocks) and training gradients are bitwise the same."""
import numpy as np
import pytest

import test_gpu_surrogate as T

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps,batch", [(1, 32), (7, 77), (40, 500)])
def test_trained_copy_is_the_loaded_one(steps, batch):
    import nqcd_mi355x as N
    from nqcd_mi355x import _lib as L
    X = T._configs(500, 3)
    Y = N.DiatomSurface().potential(X)
    E = L.Ensemble(0)
    E.surrogate_train(X, Y, steps=steps, batch=batch, lr=3e-3, lr_final=1e-4)
    for k in range(2):
        trained = E.surrogate_eval(k, X) + E.surrogate_gradient(k, X, Y)
        assert all(np.isfinite(a).all() for a in trained)
        E.surrogate_set_params(k, *E.surrogate_get_params(k))
        for a, b in zip(trained, E.surrogate_eval(k, X) + E.surrogate_gradient(k, X, Y)):
            assert np.array_equal(a, b)
    E.close()
