"""Small launches of tet vertices score every candidate on 4 waves per vertex,
larger ones take the one-wave search with its filters (csrc/dmo_kernels.hip,
line at 1,024 vertices): positions bit-exact against the oracle on meshes with
colour classes on both sides of the line, on exact and near ties, inverted
rings, scales and both nq that have the wide form."""
import numpy as np
import pytest

from test_gpu_learned_oracle import oracle_learned
from volumesurfacediscretemeshoptimization_amd import DMOMeshTetFactory, DMOTetClass, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq", [8, 4])
@pytest.mark.parametrize("jitter,scale", [(0.0, 1.0), (1e-6, 1.0), (0.3, 1.0), (0.49, 1.0), (0.3, 1e-12), (0.3, 1e5)])
def test_classes_on_both_sides(oracle, nq, jitter, scale):
    xyz, cells = synth.tet_cube(22, seed=33, jitter=jitter)
    xyz = (xyz * np.float32(scale)).astype(np.float32)
    g = DMOMeshTetFactory.create(xyz, cells)
    sizes = np.diff(g.color_offsets("inner"))
    assert sizes.min() < 1024 < sizes.max()
    opt = DMOTetClass(g, n_iter=2, nq=nq, fixed_boundary=True, quality_guard=False)
    o = oracle.OracleMesh("tet", xyz, cells)
    try:
        for it in range(2):
            opt.doIteration()
            o.iterate(nq=nq)
            gp, op = g.positions(original_order=False), o.positions()
            bad = (gp.view(np.uint32) != op.view(np.uint32)).any(axis=1)
            assert not bad.any(), (it, int(bad.sum()), np.nonzero(bad)[0][:5])
    finally:
        opt.close()
        g.close()


def test_lists_beside_windows(oracle):
    """deferred fallback lists of classes on both sides of 4,096 vertices, up
    to which a short list takes 4 waves per vertex"""
    xyz, cells = synth.tet_cube(34, seed=35, jitter=0.3)
    ref, fb = oracle_learned(oracle, "tet", xyz, cells, None, 2, 1, 0.25, "deferred", 3)
    m = DMOMeshTetFactory.create(xyz, cells)
    sizes = np.diff(m.color_offsets("inner"))
    assert sizes.min() < 4096 < sizes.max()
    o = DMOTetClass(m, n_iter=3, fixed_boundary=True, quality_guard=False)
    try:
        o.set_proposal(None, mode=2, depth=1, window_frac=0.25, fallback="deferred")
        for it in range(3):
            o.iterate(1)
            gp = m.positions(original_order=False)
            bad = (gp.view(np.uint32) != ref[it].view(np.uint32)).any(axis=1)
            assert not bad.any(), (it, int(bad.sum()), np.nonzero(bad)[0][:5])
        assert o.stats()["fallbacks"] == fb > 0
    finally:
        o.close()
        m.close()
