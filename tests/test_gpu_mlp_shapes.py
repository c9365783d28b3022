"""Surrogate inference cuts small calls finer than large ones (two members at
a time, two of the six tangent planes per workgroup).  A row's result does not
depend on the call it is in, so every size gives the rows of one large call bit
for bit; the large call is checked against the oracle in test_gpu_mlp.py.

Training takes 64 or 32 samples per workgroup, by the samples of all members
together: the gradient of a member is the same bits either way, and the
oracle's within the tolerances that test_gpu_mlp.py derives."""
import numpy as np
import pytest

import mumfim_amd as m
from oracle import mlp_oracle as mo

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


@pytest.mark.parametrize("batch", [256, 4096, 4352, 16384])
def test_gradient_of_wide_and_narrow_tiles(batch):
    rng = np.random.default_rng(batch)
    norm = (rng.normal(0, 0.1, 10).astype(np.float32), rng.uniform(0.5, 2, 10).astype(np.float32),
            rng.normal(0, 0.1, 6).astype(np.float32), rng.uniform(0.5, 2, 6).astype(np.float32))
    X = rng.normal(0, 1, (batch, 10)).astype(np.float32)
    Y = rng.normal(0, 1, (batch, 6)).astype(np.float32)
    Xd, Yd = m.DeviceArray.from_host(X), m.DeviceArray.from_host(Y)
    got = []
    for members in (4, 1):  # member 0 of both starts from the same weights
        mlp = m.SurrogateMLP(members, 7)
        mlp.set_normalization(*norm)
        got.append(mlp.gradient(0, Xd, Yd, batch))
        P = mlp.get_weights(0)
    assert got[0][0] == got[1][0]
    np.testing.assert_array_equal(got[0][1], got[1][1])
    loss, g = got[0]
    lo, go = mo.loss_and_grad(P, mo.Norm(*norm), X, Y, emulate=True)
    assert abs(loss - lo) <= 1e-4 * lo
    ends = [mo.OFF_W1, mo.OFF_B1, mo.OFF_W2, mo.OFF_B2, mo.OFF_W3, mo.OFF_B3, mo.OFF_W4,
            mo.OFF_B4, mo.NUM_PARAMS]
    for a, b in zip(ends, ends[1:]):
        assert np.linalg.norm(g[a:b] - go[a:b]) <= 2e-3 * np.linalg.norm(go[a:b])
