"""A batch whose parameters change runs the plan that a batch created with them
would run: how many solves a launch holds, and with it how wide the workgroups
of a small FP32c batch are, follows the mode and the tangent's scheme and
precision."""
import numpy as np
import pytest

import mumfim_amd as m

pytestmark = pytest.mark.gpu

CENTRAL32 = dict(tangent_precision=m.MF_PREC_FP32C, tangent_scheme=m.MF_TANGENT_CENTRAL)
SINGLE = dict(tangent_precision=m.MF_PREC_FP64, tangent_scheme=m.MF_TANGENT_FORWARD)
RELAX = dict(mode=m.MF_MODE_RELAX)
RAMP = dict(mode=m.MF_MODE_RAMP)


def make(R, **kw):
    kw.setdefault("mode", m.MF_MODE_RAMP)
    p = m.default_params(n_steps=60, precision=m.MF_PREC_FP32C, reaction_policy=1, max_steps=300,
                         **kw)
    gen = m.default_gen_params(seed=3, n_nodes=180, nonlinear_fraction=0.5)
    return m.BatchedFiberRVEAnalysisExplicit(params=p, generated=(gen, R))


def kernels(b):
    return np.asarray(b.plan()[1])[:, :3]


@pytest.mark.parametrize("first,then", [(SINGLE, CENTRAL32), (CENTRAL32, SINGLE), (RAMP, RELAX),
                                        (RELAX, RAMP)])
def test_changed_parameters_replan(first, then):
    R = 200  # one solve per RVE: wide workgroups; 13: narrow ones
    fresh, b = make(R, **then), make(R, **first)
    assert not np.array_equal(kernels(b), kernels(fresh))
    b.set_params(**then)
    np.testing.assert_array_equal(kernels(b), kernels(fresh))
    F = np.tile(np.diag([1.01, 1.0, 0.995]), (R, 1, 1))
    np.testing.assert_array_equal(b.run(F), fresh.run(F))
