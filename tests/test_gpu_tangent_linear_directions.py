"""Both tangent-linear kernels on the same networks: small batches take one
direction per workgroup, large ones three.  The plan says which kernel a batch
takes, so that each is compared with the oracle's FP64 tangent-linear (FP32c bar)
on the edges of its shapes, reaction tables, one reaction, no free node, and a
second update run from the committed state; the copies of a network in a large
batch give the same bits."""
import numpy as np
import pytest

import mumfim_amd as mf
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

TOL = 1e-4  # FP32c stress and tangent against FP64


def strain(seed, n, amp):
    u = np.random.default_rng(seed).uniform(-amp, amp, (n, 3, 3))
    return np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1))


def rel(a, b):
    a, b = np.asarray(a).reshape(len(a), -1), np.asarray(b).reshape(len(b), -1)
    return float((np.abs(a - b).max(1) / np.abs(b).max(1)).max())


def networks(kind):
    if isinstance(kind, tuple):
        return [mf.generate_network(seed=500 + n, n_nodes=n, nonlinear_fraction=0.5)
                for n in kind]
    net = mf.generate_network(seed=88, n_nodes=330, nonlinear_fraction=0.5)
    if kind == "table":
        stiff = mf.Reaction(mf.MF_REACTION_NONLINEAR, 3.0e-8, 9.0e7, 900.0, 2.0, 1.02, 0.99)
        net.reactions = net.reactions + [stiff]
        net.fiber_reaction = np.arange(net.n_fibers, dtype=np.int32) % 3
    elif kind == "one linear reaction":
        net.reactions, net.fiber_reaction = net.reactions[:1], np.zeros(net.n_fibers, np.int32)
    elif kind == "one toe reaction":
        net.reactions, net.fiber_reaction = net.reactions[1:], np.zeros(net.n_fibers, np.int32)
    else:
        net.boundary = np.arange(net.n_nodes, dtype=np.int32)
    return [net]


KINDS = ["table", "one linear reaction", "one toe reaction", "no free node",
         (20, 286, 290, 294), (573, 580, 586), (865, 872, 1730, 1742, 2150)]


@pytest.mark.parametrize("dirs", [1, 3])
@pytest.mark.parametrize("kind", KINDS, ids=str)
def test_both_kernels(kind, dirs):
    print(f"case: {kind}, {dirs} directions", flush=True)
    nets = networks(kind)
    n = len(nets)
    # six workgroups of one direction per RVE and at least 129 RVEs: beyond every
    # room that the planner gives them (three of 256 threads per CU)
    copies = -(-129 // n) if dirs == 3 else 1
    p = mf.default_params(mode=mf.MF_MODE_RAMP, n_steps=300, precision=mf.MF_PREC_FP32C,
                          reaction_policy=mf.MF_REACT_PER_FIBER,
                          tangent_scheme=mf.MF_TANGENT_LINEAR,
                          tangent_precision=mf.MF_PREC_FP32C)
    g, o = mf.BatchedFiberRVEAnalysisExplicit(nets * copies, p), Oracle(nets, p)
    assert (g.tangent_plan()[:, 2] == dirs).all(), g.tangent_plan()[:n]
    for seed, amp in ((1, 0.05), (2, 0.02)):
        F = strain(seed, n, amp)
        s, C, st = g.run_with_tangent(np.tile(F, (copies, 1, 1)), return_status=True)
        so, Co = o.run(F), o.computeMaterialStiffness()
        s, C = np.asarray(s).reshape(copies, n, 6), np.asarray(C).reshape(copies, n, 36)
        print(f"  sigma {rel(s[0], so):.2e} C {rel(C[0], Co):.2e}", flush=True)
        assert (st == mf.MF_STATUS_OK).all()
        assert rel(s[0], so) <= TOL and rel(C[0], Co) <= TOL
        assert (s == s[0]).all() and (C == C[0]).all()
    g.close()
