"""The tangent-linear kernel with three directions per workgroup at the edges
of its shapes (free nodes around a thread count and its multiples, RVEs at and
beyond its LDS, reaction tables, no free node), against the oracle's FP64
tangent-linear with the FP32c bar; a second update run checks the committed
state."""
import sys

import numpy as np
import pytest

import mumfim_amd as mf
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-4  # FP32c stress and tangent against FP64


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def strain(seed, n, amp):
    u = np.random.default_rng(seed).uniform(-amp, amp, (n, 3, 3))
    return np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1))


def rel(a, b):
    a, b = np.asarray(a).reshape(len(a), -1), np.asarray(b).reshape(len(b), -1)
    return float((np.abs(a - b).max(1) / np.abs(b).max(1)).max())


def check(nets, steps=300):
    p = mf.default_params(mode=mf.MF_MODE_RAMP, n_steps=steps, precision=mf.MF_PREC_FP32C,
                          reaction_policy=mf.MF_REACT_PER_FIBER,
                          tangent_scheme=mf.MF_TANGENT_LINEAR,
                          tangent_precision=mf.MF_PREC_FP32C)
    g, o = mf.BatchedFiberRVEAnalysisExplicit(nets, p), Oracle(nets, p)
    for seed, amp in ((1, 0.05), (2, 0.02)):
        F = strain(seed, len(nets), amp)
        s, C, st = g.run_with_tangent(F, return_status=True)
        so = o.run(F)
        Co = o.computeMaterialStiffness()
        say(f"  sigma {rel(s, so):.2e} C {rel(C, Co):.2e}")
        assert (st == mf.MF_STATUS_OK).all()
        assert rel(s, so) <= TOL and rel(C, Co) <= TOL


@pytest.mark.parametrize("law", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("sizes", [[20, 286, 290, 294], [573, 580, 586], [865, 872, 1730, 1742],
                                   [2150, 2250]])
def test_shapes(sizes, law):
    say(f"case: sizes {sizes} law {law}")
    check([mf.generate_network(seed=500 + n, n_nodes=n, nonlinear_fraction=law) for n in sizes])


@pytest.mark.parametrize("kind", ["table", "no free node"])
def test_tables_and_boundaries(kind):
    say(f"case: {kind}")
    net = mf.generate_network(seed=88, n_nodes=330, nonlinear_fraction=0.5)
    if kind == "table":
        stiff = mf.Reaction(mf.MF_REACTION_NONLINEAR, 3.0e-8, 9.0e7, 900.0, 2.0, 1.02, 0.99)
        net.reactions = net.reactions + [stiff]
        net.fiber_reaction = np.arange(net.n_fibers, dtype=np.int32) % 3
    else:
        net.boundary = np.arange(net.n_nodes, dtype=np.int32)
    check([net, net])


@pytest.mark.parametrize("law", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("sizes", [[20, 286, 290, 294], [573, 580, 586], [865, 872, 1730, 1742],
                                   [2150, 2250]])
def test_few_and_many(sizes, law):
    """Small batches take one direction per workgroup, large ones three: the
    same trajectory and derivatives, so stress and tangent agree up to the order
    of their FP64 sums over the boundary nodes, which follows the thread count."""
    say(f"case: few and many, sizes {sizes} law {law}")
    nets = [mf.generate_network(seed=500 + n, n_nodes=n, nonlinear_fraction=law) for n in sizes]
    p = mf.default_params(mode=mf.MF_MODE_RAMP, n_steps=120, precision=mf.MF_PREC_FP32C,
                          reaction_policy=mf.MF_REACT_PER_FIBER,
                          tangent_scheme=mf.MF_TANGENT_LINEAR,
                          tangent_precision=mf.MF_PREC_FP32C)
    F = strain(3, len(nets), 0.05)
    few = mf.BatchedFiberRVEAnalysisExplicit(nets, p)
    copies = 132 // len(nets)  # more than 128 RVEs: beyond both lines
    many = mf.BatchedFiberRVEAnalysisExplicit(nets * copies, p)
    s1, C1 = few.run_with_tangent(F)
    s3, C3 = many.run_with_tangent(np.tile(F, (copies, 1, 1)))
    n = len(nets)
    for k in (0, copies - 1):
        for many_, few_ in ((C3, C1), (s3, s1)):
            np.testing.assert_allclose(np.asarray(many_)[k * n:(k + 1) * n], few_, rtol=0,
                                       atol=1e-13 * np.abs(few_).max())
