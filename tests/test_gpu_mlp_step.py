"""The fused training step (csrc/mlp.hip: k_mlp_rows, k_mlp_grads): gradients at
row counts around its tiles of 16 rows, MFMA depth of 32 and sums of 256
against the FP64 restatement (the bars of test_gpu_learned.py), a training step
against Adam applied to the same rows' gradients, and the transposed copy of W2
that the step keeps.
"""
import numpy as np
import pytest

import mlp_ref
from volumesurfacediscretemeshoptimization_amd import DMODataset, DMOMeshTetFactory, DMOMLP, DMOTetClass, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 255, 256, 257, 513, 2049])
def test_gradients_at_tile_edges(n):
    rng = np.random.default_rng(n)
    X = (rng.normal(size=(n, 96)) * 0.6).astype(np.float32)
    T = (rng.normal(size=(n, 3)) * 0.1).astype(np.float32)
    mlp = DMOMLP(seed=9)
    p = mlp.params().astype(np.float64)
    loss, g = mlp.gradients(X, T)
    lr_, gr = mlp_ref.loss_and_grad(p, X, T, emulate=True)
    assert abs(loss - lr_) <= 1e-3 * abs(lr_)
    for name, sl in mlp_ref.block_slices().items():
        rel = np.linalg.norm(g[sl].astype(np.float64) - gr[sl]) / np.linalg.norm(gr[sl])
        assert rel < 3e-2, (n, name, rel)
    mlp.close()


def _shuffle(n, seed):
    """the training epoch's permutation (SplitMix64, Fisher-Yates from the end)"""
    m64, s, p = (1 << 64) - 1, seed, list(range(n))
    for i in range(n - 1, 0, -1):
        s = (s + 0x9e3779b97f4a7c15) & m64
        z = ((s ^ (s >> 30)) * 0xbf58476d1ce4e5b9) & m64
        z = ((z ^ (z >> 27)) * 0x94d049bb133111eb) & m64
        j = (z ^ (z >> 31)) % (i + 1)
        p[i], p[j] = p[j], p[i]
    return p


def test_training_step_is_adam_on_the_batch_gradient():
    xyz, tets = synth.tet_cube(8, seed=5)
    m = DMOMeshTetFactory.create(xyz, tets)
    o = DMOTetClass(m, n_iter=1, fixed_boundary=True)
    ds = DMODataset(343)
    o.record(ds, 1)
    n = len(ds)
    X, T = ds.get(0, n)
    perm = _shuffle(n, 5)
    a, b = DMOMLP(seed=1), DMOMLP(seed=1)
    w0 = a.params()
    loss, g = b.gradients(X[perm], T[perm])
    el = a.train(ds, epochs=1, batch=n, lr=1e-3, seed=5)
    assert el[0] == loss
    f = np.float32
    m1 = (f(1) - f(0.9)) * g
    m2 = (f(1) - f(0.999)) * g * g
    step = f(1e-3) * (m1 / (f(1) - f(0.9))) / (np.sqrt(m2 / (f(1) - f(0.999))) + f(1e-8))
    # the update is computed in FP32 in this order: a few roundings of it and one of w
    assert np.all(np.abs(a.params() - (w0 - step)) <= 4e-7 * np.abs(step) + 6e-8 * np.abs(w0))
    # the backward pass of the trained network reads the same weights as one set from its parameters
    a.train(ds, epochs=3, batch=64, lr=1e-3, seed=6)
    b.set_params(a.params())
    la, ga = a.gradients(X, T)
    lb, gb = b.gradients(X, T)
    assert la == lb and np.array_equal(ga, gb)
    for x in (o, m, ds, a, b):
        x.close()
