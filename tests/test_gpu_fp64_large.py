"""The FP64 kernels of large and dense RVEs bit for bit: the node-centric kernel
without range handling (solve64n) against the energy-tracking kernel, which keeps
the compiler's IEEE operations, in each of its shapes, and against the oracle's
state; the kernel with t records (solve64t) with more than two laws; and that
unusual tables and degrees run the fiber-once kernel that they are a test of."""
import numpy as np
import pytest

import mumfim_amd as mf
from oracle.oracle import Oracle

pytestmark = pytest.mark.gpu

LINEAR = mf.Reaction(mf.MF_REACTION_LINEAR, 3.5e-8, 4.32e7, 1000.0)
TOE = mf.Reaction(mf.MF_REACTION_NONLINEAR, 3.5e-8, 4.32e7, 1000.0, 1.2, 1.05, 1.0)
STIFF = mf.Reaction(mf.MF_REACTION_NONLINEAR, 3.0e-8, 9.0e7, 900.0, 2.0, 1.02, 0.99)
ONCE, FAST = 16384, 65536  # fiber-once; fast64 RVEs beyond its force records


def strain(n, amp, seed=3):
    u = np.random.default_rng(seed).uniform(-amp, amp, (n, 3, 3))
    return np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1))


def run(nets, F, **kw):
    g = mf.BatchedFiberRVEAnalysisExplicit(
        nets, mf.default_params(reaction_policy=mf.MF_REACT_PER_FIBER, **kw))
    plan = g.plan()[1][:, :3].tolist()
    s, st = g.run(F, return_status=True)
    x, u, _ = g.get_state()
    g.close()
    return plan, (s, st, x, u)


def same_bits(nets, flag, F, slots=None, **kw):
    plan, fast = run(nets, F, **kw)
    print(f"  plan {plan}", flush=True)
    assert all(f & (ONCE | FAST) == flag for _, _, f in plan), plan
    assert slots is None or [s for _, s, _ in plan] == slots
    eplan, ref = run(nets, F, energy_diagnostics=1, **kw)
    assert not any(f & (ONCE | FAST) for _, _, f in eplan), eplan
    for a, b in zip(fast, ref):
        assert np.array_equal(a, b)


# one law and ~9 fibers per node: the t records leave LDS at two, three and four
# nodes per thread
@pytest.mark.parametrize("law", [0.0, 1.0])
@pytest.mark.parametrize("mode", [mf.MF_MODE_RAMP, mf.MF_MODE_RELAX])
def test_node_centric_shapes(law, mode):
    print(f"case: law {law} mode {mode}", flush=True)
    nets = [mf.generate_network(seed=60 + n, n_nodes=n, nonlinear_fraction=law, k_neighbors=14)
            for n in (2000, 2600, 3600)]
    kw = dict(mode=mode, n_steps=230)
    if mode == mf.MF_MODE_RELAX:
        kw.update(tolerance=1e-30, max_steps=205)
    same_bits(nets, FAST, strain(3, 0.1), slots=[2, 3, 4], **kw)


@pytest.mark.parametrize("mode", [mf.MF_MODE_RAMP, mf.MF_MODE_RELAX])
def test_node_centric_state_is_the_oracles(mode):
    """Linear fibers (the toe law's exponential is the host library's there)."""
    print(f"case: oracle, mode {mode}", flush=True)
    nets = [mf.generate_network(seed=300 + n, n_nodes=n) for n in (3900, 4300)]
    kw = dict(mode=mode, n_steps=230)
    if mode == mf.MF_MODE_RELAX:
        kw.update(tolerance=1e-30, max_steps=205)
    F = strain(2, 0.1)
    plan, (s, st, x, u) = run(nets, F, **kw)
    assert all(f & (ONCE | FAST) == FAST for _, _, f in plan), plan
    o = Oracle(nets, mf.default_params(reaction_policy=mf.MF_REACT_PER_FIBER, **kw))
    so, sto = o.run(F, return_status=True)
    xo, uo, _ = o.get_state()
    assert np.array_equal(st, sto)
    assert np.array_equal(x, xo) and np.array_equal(u, uo)
    assert np.abs(s - so).max() <= 1e-10 * np.abs(so).max()


@pytest.mark.parametrize("n", [2330, 3500])
def test_t_records_with_three_reactions(n):
    print(f"case: three reactions, {n} nodes", flush=True)
    net = mf.generate_network(seed=9, n_nodes=n)
    net.reactions = [TOE, LINEAR, STIFF]
    net.fiber_reaction = np.arange(net.n_fibers, dtype=np.int32) % 3
    same_bits([net], ONCE | FAST, strain(1, 0.1), mode=mf.MF_MODE_RAMP, n_steps=230)


@pytest.mark.parametrize("kind", ["three reactions", "two linear", "hub", "no free node"])
def test_unusual_tables_and_degrees_run_fiber_once(kind):
    print(f"case: {kind}", flush=True)
    net = mf.generate_network(seed=77, n_nodes=330, nonlinear_fraction=0.5)
    if kind == "three reactions":
        net.reactions = [LINEAR, TOE, STIFF]
        net.fiber_reaction = np.arange(net.n_fibers, dtype=np.int32) % 3
    elif kind == "two linear":
        net.reactions = [LINEAR, mf.Reaction(mf.MF_REACTION_LINEAR, 5.0e-8, 2.0e7, 1000.0)]
    elif kind == "hub":  # one node with more fibers than any register list
        free = np.setdiff1d(np.arange(net.n_nodes), net.boundary)
        have = {tuple(sorted(f)) for f in net.fibers.tolist()}
        new = [(free[0], r) for r in free[1:31] if tuple(sorted((free[0], r))) not in have]
        net.fibers = np.concatenate([net.fibers, np.array(new, np.int32)])
        net.fiber_reaction = np.concatenate([net.fiber_reaction,
                                             np.zeros(len(new), np.int32)])
    else:
        net.boundary = np.arange(net.n_nodes, dtype=np.int32)
    same_bits([net, net], ONCE, strain(2, 0.08), mode=mf.MF_MODE_RAMP, n_steps=150,
              block_size=512)
