"""Surrogate inference cuts small calls finer than large ones (two members at
a time, two of the six tangent planes per workgroup).  A row's result does not
depend on the call it is in, so every size gives the rows of one large call bit
for bit; the large call is checked against the oracle in test_gpu_mlp.py."""
import numpy as np
import pytest

import mumfim_amd as m

pytestmark = pytest.mark.gpu

N_MAX = 4200  # beyond both lines: 1360 rows with a Jacobian, 4096 without


@pytest.fixture(scope="module", params=[1, 2, 3, 4])
def ensemble(request):
    rng = np.random.default_rng(request.param)
    mlp = m.SurrogateMLP(request.param, 7)
    X = rng.normal(size=(N_MAX, 10)).astype(np.float32)
    mlp.set_normalization(rng.normal(0, 0.1, 10), rng.uniform(0.5, 2.0, 10),
                          rng.normal(0, 0.1, 6), rng.uniform(0.5, 2.0, 6))
    return mlp, X, mlp.predict(X), mlp.predict(X, jacobian=True)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 777, 1360, 1361, 4096, 4097])
def test_rows_do_not_depend_on_the_size_of_the_call(ensemble, n):
    mlp, X, (Y0, S0, _), (Y1, S1, J1) = ensemble
    # rows from the end, so that each row meets another place in its tile
    Y, S, _ = mlp.predict(X[N_MAX - n:])
    np.testing.assert_array_equal(Y, Y0[N_MAX - n:])
    np.testing.assert_array_equal(S, S0[N_MAX - n:])
    Y, S, J = mlp.predict(X[N_MAX - n:], jacobian=True)
    np.testing.assert_array_equal(Y, Y1[N_MAX - n:])
    np.testing.assert_array_equal(S, S1[N_MAX - n:])
    np.testing.assert_array_equal(J, J1[N_MAX - n:])


def test_one_member_of_an_ensemble_small_and_large(ensemble):
    mlp, X, _, _ = ensemble
    for k in range(mlp.n_members):
        Y0, _, J0 = mlp.predict(X, jacobian=True, member=k)
        Y, _, J = mlp.predict(X[:100], jacobian=True, member=k)
        np.testing.assert_array_equal(Y, Y0[:100])
        np.testing.assert_array_equal(J, J0[:100])
