"""The arrays that only the streaming FP64 kernels read are there for the batches
that run them and for no others: the device memory of a batch, FP64 tangents of
an FP32c batch, and a batch switched to FP64 after its creation."""
import ctypes as C

import numpy as np
import pytest

import mumfim_amd as mf

pytestmark = pytest.mark.gpu

MB = 1 << 20


def free_bytes():
    f, t = C.c_size_t(), C.c_size_t()
    assert mf.lib().hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def batch(n_nodes, R, prec, law=0.5, **kw):
    kw.setdefault("tangent_precision", prec)
    p = mf.default_params(mode=mf.MF_MODE_RAMP, n_steps=40, precision=prec,
                          reaction_policy=mf.MF_REACT_PER_FIBER, **kw)
    gen = mf.default_gen_params(seed=31, nonlinear_fraction=law, n_nodes=n_nodes)
    return mf.BatchedFiberRVEAnalysisExplicit(params=p, generated=(gen, R))


def footprint(*args):
    before = free_bytes()
    b = batch(*args)
    used = before - free_bytes()
    flags = {int(f) & (16384 | 65536) for f in b.plan()[1][:, 2]}
    b.close()
    return used, flags


def test_memory_follows_the_kernels():
    print("case: memory", flush=True)
    batch(60, 1, mf.MF_PREC_FP64).close()  # module and runtime are up
    # 250 RVEs of 2300 nodes: ~6600 fibers each, 20 bytes a fiber streamed
    large = 20 * 250 * mf.generate_network(seed=31, n_nodes=2300).n_fibers
    f32, _ = footprint(2300, 250, mf.MF_PREC_FP32C)
    f64, flags = footprint(2300, 250, mf.MF_PREC_FP64)
    assert flags == {16384 | 65536}
    print(f"  2300 nodes: FP32c {f32 / MB:.1f} MB, FP64 {f64 / MB:.1f} MB", flush=True)
    assert f64 - f32 >= 0.9 * large
    # 1500 RVEs of 400 nodes: the fiber-once kernel's own tables are all it needs
    f32, _ = footprint(400, 1500, mf.MF_PREC_FP32C)
    f64, flags = footprint(400, 1500, mf.MF_PREC_FP64)
    assert flags == {16384}
    print(f"  400 nodes: FP32c {f32 / MB:.1f} MB, FP64 {f64 / MB:.1f} MB", flush=True)
    assert abs(f64 - f32) <= 8 * MB


# RVEs with t records, and single-law ones beyond them (node-centric)
@pytest.mark.parametrize("n_nodes,law,flag", [(2300, 0.5, 16384 | 65536), (4000, 0.0, 65536)])
def test_fp64_use_of_an_fp32_batch(n_nodes, law, flag):
    print(f"case: {n_nodes} nodes, law {law}", flush=True)
    F = np.diag([1.02, 0.99, 1.01])[None].repeat(2, 0)
    g = batch(n_nodes, 2, mf.MF_PREC_FP64, law)
    assert all(int(f) & (16384 | 65536) == flag for f in g.plan()[1][:, 2])
    s64 = g.run(F)
    C64 = g.computeMaterialStiffness()
    g.close()
    # the first update run starts from the reference state in either precision, so
    # the FP64 differences around it are the same solves
    g = batch(n_nodes, 2, mf.MF_PREC_FP32C, law, tangent_precision=mf.MF_PREC_FP64)
    g.run(F)
    assert np.array_equal(g.computeMaterialStiffness(), C64)
    g.close()
    g = batch(n_nodes, 2, mf.MF_PREC_FP32C, law)
    g.set_params(precision=mf.MF_PREC_FP64)
    assert np.array_equal(g.run(F), s64)
    g.close()
