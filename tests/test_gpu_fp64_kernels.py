"""The FP64 fiber-once and large-RVE kernels against the node-centric kernel
that tracks energies (which keeps the compiler's IEEE square roots and
divisions): the same bits at the edges of their shapes.  Also their
range-free square root and quotient behind it, through solves whose lengths and
forces they round, and the networks that must not take them."""
import sys

import numpy as np
import pytest

import mumfim_amd as mf

pytestmark = pytest.mark.gpu

LINEAR = mf.Reaction(mf.MF_REACTION_LINEAR, 3.5e-8, 4.32e7, 1000.0)
TOE = mf.Reaction(mf.MF_REACTION_NONLINEAR, 3.5e-8, 4.32e7, 1000.0, 1.2, 1.05, 1.0)


def say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


def strain(n, amp, seed=3):
    u = np.random.default_rng(seed).uniform(-amp, amp, (n, 3, 3))
    return np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1))


def both(nets, F, **kw):
    """sigma and state of a committed run on the planner's kernels and on the
    energy-tracking one."""
    out = []
    for en in (0, 1):
        g = mf.BatchedFiberRVEAnalysisExplicit(
            nets, mf.default_params(energy_diagnostics=en,
                                    reaction_policy=mf.MF_REACT_PER_FIBER, **kw))
        flags = [int(f) for f in g.plan()[1][:, 2]]
        s, st = g.run(F, return_status=True)
        x, u, _ = g.get_state()
        out.append((s, st, x, u))
        say(f"  plan {sorted(set(map(tuple, g.plan()[1][:, :3].tolist())))}")
        if en == 0:
            fast = [f & (16384 | 65536) for f in flags]
        g.close()
    return out[0], out[1], fast


# free nodes just below and above a thread count and its double, fibers beyond
# the lanes' registers, and RVEs whose force records leave LDS
@pytest.mark.parametrize("law", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("sizes", [[8, 40, 286, 290, 296], [570, 579, 585], [1150, 1162, 1800],
                                   [1850, 2300, 2330], [3380, 4000]])
@pytest.mark.parametrize("mode", [mf.MF_MODE_RAMP, mf.MF_MODE_RELAX])
def test_bits_of_the_node_centric_kernel(sizes, law, mode):
    say(f"case: sizes {sizes} law {law} mode {mode}")
    nets = [mf.generate_network(seed=300 + n, n_nodes=n, nonlinear_fraction=law) for n in sizes]
    if max(sizes) > 3000:  # energies are not tracked that far: FP64 parity is the oracle's
        sizes = None
    F = strain(len(nets), 0.1)
    kw = dict(mode=mode, n_steps=230)
    if mode == mf.MF_MODE_RELAX:
        kw.update(tolerance=1e-30, max_steps=205)
    if sizes is None:
        from oracle.oracle import Oracle
        p = mf.default_params(reaction_policy=mf.MF_REACT_PER_FIBER, **kw)
        g = mf.BatchedFiberRVEAnalysisExplicit(nets, p)
        assert all(int(f) & 65536 for f in g.plan()[1][:, 2])
        s, o = g.run(F), Oracle(nets, p).run(F)
        err = np.abs(s - o).max() / np.abs(o).max()
        say(f"  vs oracle {err:.2e}")
        # mixed laws are summed nonlinear first here and in fiber order there
        assert err <= 1e-10
        return
    a, b, fast = both(nets, F, **kw)
    assert all(fast), fast
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("kind", ["three reactions", "two linear", "hub", "no free node"])
def test_bits_with_unusual_tables_and_degrees(kind):
    say(f"case: {kind}")
    net = mf.generate_network(seed=77, n_nodes=330, nonlinear_fraction=0.5)
    if kind == "three reactions":
        stiff = mf.Reaction(mf.MF_REACTION_NONLINEAR, 3.0e-8, 9.0e7, 900.0, 2.0, 1.02, 0.99)
        net.reactions = [LINEAR, TOE, stiff]
        net.fiber_reaction = np.arange(net.n_fibers, dtype=np.int32) % 3
    elif kind == "two linear":
        net.reactions = [LINEAR, mf.Reaction(mf.MF_REACTION_LINEAR, 5.0e-8, 2.0e7, 1000.0)]
    elif kind == "hub":  # one node with more fibers than any register list
        free = np.setdiff1d(np.arange(net.n_nodes), net.boundary)
        hub, rest = free[0], free[1:31]
        have = {tuple(sorted(f)) for f in net.fibers.tolist()}
        new = [(hub, r) for r in rest if tuple(sorted((hub, r))) not in have]
        net.fibers = np.concatenate([net.fibers, np.array(new, np.int32)])
        net.fiber_reaction = np.concatenate([net.fiber_reaction,
                                             np.zeros(len(new), np.int32)])
    else:
        net.boundary = np.arange(net.n_nodes, dtype=np.int32)
    # one thread count for both: the stress of more boundary nodes than threads
    # is summed in an order that follows it
    a, b, _ = both([net, net], strain(2, 0.08), mode=mf.MF_MODE_RAMP, n_steps=150,
                   block_size=512)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


def test_out_of_range_networks_keep_the_ieee_kernels():
    """Coincident nodes (a fiber of length zero) and lengths near the ends of
    the FP64 range are not for the kernels without range handling; they run,
    and report what the energy-tracking kernel reports."""
    say("case: zero-length fiber, 1e-120 cube")
    flat = mf.generate_network(seed=5, n_nodes=60)
    free = np.setdiff1d(np.arange(60), flat.boundary)
    flat.coords[free[1]] = flat.coords[free[0]]
    flat.fibers = np.concatenate([flat.fibers, np.array([[free[0], free[1]]], np.int32)])
    flat.fiber_reaction = np.append(flat.fiber_reaction, np.int32(0))
    tiny = mf.generate_network(seed=6, n_nodes=60)
    tiny.coords = tiny.coords * 1e-120
    a, b, fast = both([flat, tiny], strain(2, 0.05), mode=mf.MF_MODE_RAMP, n_steps=40)
    assert not any(fast), fast
    assert np.array_equal(a[1], b[1])
    assert np.array_equal(a[0], b[0], equal_nan=True)
