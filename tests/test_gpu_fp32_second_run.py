"""An FP32c run from a committed state is as accurate as one from the reference
state, on every shape of the register kernel: positions against the same two runs
in FP64.

Bar: displacements of up to 0.1 integrated in compensated FP32 from forces of
relative rounding ~1e-7 stay within a few 1e-8 of the cube's size (first runs
measure 1e-8 to 3e-8); 1e-6 leaves a factor of thirty."""
import numpy as np
import pytest

import mumfim_amd as mf

pytestmark = pytest.mark.gpu

# nodes, law, parameters, (threads, nodes per lane)
SHAPES = [(180, 0.0, dict(fp32_kernel=mf.MF_FP32_KERNEL_WAVE), (256, 3)),
          (150, 0.5, dict(fp32_kernel=mf.MF_FP32_KERNEL_WAVE), (64, 3)),
          (359, 0.0, dict(block_size=256), (256, 2)),
          (420, 1.0, dict(block_size=512), (512, 1)),
          (359, 0.0, dict(block_size=512), (512, 1)),
          (1000, 0.0, dict(block_size=512), (512, 3)),
          (1700, 0.0, dict(block_size=512), (512, 4)),
          (1000, 0.0, dict(block_size=768), (768, 2)),
          (900, 0.5, dict(block_size=512, fp32_kernel=mf.MF_FP32_KERNEL_NODE), (512, 3))]


def two_runs(net, mode, **kw):
    p = mf.default_params(mode=mode, n_steps=60, max_steps=60, tolerance=1e-30,
                          reaction_policy=mf.MF_REACT_PER_FIBER, **kw)
    g = mf.BatchedFiberRVEAnalysisExplicit([net], p)
    plan = g.plan()[1][0, :3].tolist()
    xs = []
    for seed in (5, 6):
        u = np.random.default_rng(seed).uniform(-0.08, 0.08, (1, 3, 3))
        g.run(np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1)))
        xs.append(g.get_state()[0])
    g.close()
    return plan, xs


@pytest.mark.parametrize("mode", [mf.MF_MODE_RAMP, mf.MF_MODE_RELAX])
@pytest.mark.parametrize("n,law,kw,shape", SHAPES, ids=str)
def test_second_run(n, law, kw, shape, mode):
    print(f"case: {n} nodes law {law} {kw} mode {mode}", flush=True)
    net = mf.generate_network(seed=13210, n_nodes=n, nonlinear_fraction=law)
    plan, x32 = two_runs(net, mode, precision=mf.MF_PREC_FP32C, **kw)
    print(f"  plan {plan}", flush=True)
    assert tuple(plan[:2]) == shape and plan[2] & 4  # lists in registers
    _, x64 = two_runs(net, mode, precision=mf.MF_PREC_FP64)
    err = [float(np.abs(a - b).max()) for a, b in zip(x32, x64)]
    print(f"  error of the positions: first {err[0]:.2e}, second {err[1]:.2e}", flush=True)
    assert err[0] <= 1e-6 and err[1] <= 1e-6


@pytest.mark.parametrize("n,law", [(130, 0.5), (180, 0.0), (250, 0.0), (400, 1.0)])
def test_second_run_does_not_depend_on_the_size_of_its_batch(n, law):
    """Small batches run a node per lane, large ones several: the same bits."""
    print(f"case: {n} nodes law {law}", flush=True)
    net = mf.generate_network(seed=77, n_nodes=n, nonlinear_fraction=law)
    p = mf.default_params(mode=mf.MF_MODE_RAMP, n_steps=60, precision=mf.MF_PREC_FP32C,
                          reaction_policy=mf.MF_REACT_PER_FIBER)
    got = []
    for R in (1, 1100):
        g = mf.BatchedFiberRVEAnalysisExplicit([net] * R, p)
        for seed in (5, 6):
            u = np.random.default_rng(seed).uniform(-0.08, 0.08, (1, 3, 3))
            g.run(np.repeat(np.eye(3)[None] + 0.5 * (u + u.transpose(0, 2, 1)), R, 0))
        got.append((g.plan()[1][0, :3].tolist(), g.get_state()[0][:n]))
        g.close()
    assert got[0][0] != got[1][0]  # different kernels
    np.testing.assert_array_equal(got[0][1], got[1][1])
