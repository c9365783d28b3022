"""Small FP32c ramp batches run on wider workgroups (a node per thread) than
large ones.  Every node's sums keep their order, so a solve gives the same
result in a batch of any size: the positions bit for bit, the stress up to the
order in which its FP64 contributions are added (a few units in the last place
of the largest component, here 1e-13 of it)."""
import numpy as np
import pytest

import mumfim_amd as m

pytestmark = pytest.mark.gpu

F = np.diag([1.03, 0.99, 1.01])


def solve(n_nodes, toe, R, **kw):
    p = m.default_params(mode=m.MF_MODE_RAMP, n_steps=60, precision=m.MF_PREC_FP32C,
                         reaction_policy=1, **kw)
    gen = m.default_gen_params(seed=3, nonlinear_fraction=toe, n_nodes=n_nodes)
    b = m.BatchedFiberRVEAnalysisExplicit(params=p, generated=(gen, R))
    plan = np.asarray(b.plan()[1])
    sigma = np.asarray(b.run(np.tile(F, (R, 1, 1)), update_coords=False))
    b.close()
    return sigma, plan[:, :3]


@pytest.mark.parametrize("toe", [0.0, 0.5])
@pytest.mark.parametrize("n_nodes", [130, 180, 250, 400])
def test_a_solve_does_not_depend_on_the_size_of_its_batch(n_nodes, toe):
    ref, narrow = solve(n_nodes, toe, 1025)
    scale = np.abs(ref).max(axis=1, keepdims=True)
    for R in (1, 256, 257, 512, 513, 1024):
        sigma, plan = solve(n_nodes, toe, R)
        assert np.all(np.abs(sigma - ref[:R]) <= 1e-13 * scale[:R]), R
        assert np.all(plan[:, 1] <= narrow[:R, 1])  # never more nodes per thread


def test_differenced_fp32_tangents_count_all_their_solves():
    """A tangent by FP32c central differences launches 13 solves per RVE: its
    batches keep the narrow workgroups from 79 RVEs on."""
    kw = dict(tangent_precision=m.MF_PREC_FP32C, tangent_scheme=m.MF_TANGENT_CENTRAL)
    _, one = solve(180, 0.0, 80)
    _, many = solve(180, 0.0, 80, **kw)
    _, narrow = solve(180, 0.0, 1025)
    assert np.all(one[:, 1] == 1)
    np.testing.assert_array_equal(many, narrow[:80])
