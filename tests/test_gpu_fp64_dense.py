"""FP64 RVEs with more fibers than a forced thread count holds in registers
still evaluate each fiber once, with the bits of the node-centric kernel that
tracks energies."""
import numpy as np
import pytest

import mumfim_amd as mf

pytestmark = pytest.mark.gpu


def run(nets, F, **kw):
    g = mf.BatchedFiberRVEAnalysisExplicit(
        nets, mf.default_params(reaction_policy=mf.MF_REACT_PER_FIBER, **kw))
    plan = g.plan()[1][:, :3].tolist()
    s, st = g.run(F, return_status=True)
    x, u, _ = g.get_state()
    g.close()
    return plan, (s, st, x, u)


# fibers per thread: 256 threads hold 6, 512 threads 6, with two nodes each
@pytest.mark.parametrize("law", [0.0, 0.5, 1.0])
@pytest.mark.parametrize("block,sizes", [(256, [330, 450, 540]), (512, [640, 900, 1080])])
@pytest.mark.parametrize("mode", [mf.MF_MODE_RAMP, mf.MF_MODE_RELAX])
def test_forced_threads_with_many_fibers(block, sizes, law, mode):
    print(f"case: block {block} sizes {sizes} law {law} mode {mode}", flush=True)
    nets = [mf.generate_network(seed=40 + n, n_nodes=n, nonlinear_fraction=law, k_neighbors=8)
            for n in sizes]
    assert all(n.n_fibers > 6 * block for n in nets[1:])
    u = np.random.default_rng(6).uniform(-0.1, 0.1, (len(nets), 3, 3))
    F = np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1))
    kw = dict(mode=mode, n_steps=230, block_size=block)
    if mode == mf.MF_MODE_RELAX:
        kw.update(tolerance=1e-30, max_steps=205)
    plan, fast = run(nets, F, **kw)
    assert all(b == block and f & 16384 for b, _, f in plan), plan
    _, ref = run(nets, F, energy_diagnostics=1, **kw)
    for a, b in zip(fast, ref):
        assert np.array_equal(a, b)
