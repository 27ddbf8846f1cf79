"""The searches where their bounds leave (nearly) everything to score, and the
selection over a ring whose elements are all alike (csrc/dmo_kernels.hip,
csrc/vsdmo_numerics.h): positions bit-exact against the oracle."""
import numpy as np
import pytest

from test_gpu_search_bounds import _compare, _cube, _hex_fan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("metric", [0, 1])
@pytest.mark.parametrize("jitter", [0.0, 1e-7, 1e-4, 0.02])
def test_hex_rings_of_equal_elements(oracle, jitter, metric):
    """every ratio within rounding of the smallest: the selection goes from one
    that replaces the last to the next"""
    xyz, cells = _cube("hex", 8, 81, jitter)
    _compare(oracle, "hex", xyz, cells, hex_metric=metric)


@pytest.mark.parametrize("nq", [2, 4, 6, 8])
@pytest.mark.parametrize("jitter,grid_scale", [(0.0, 0.5), (0.02, 0.5), (0.25, 0.5), (0.25, 4.0), (0.45, 1.0)])
def test_hex_windows_wider_than_the_bounds(oracle, nq, jitter, grid_scale):
    """windows of the largest ring offset: none to all of the 40 (32) sub-tets
    are left to a level, odd and even numbers of them"""
    xyz, cells = _cube("hex", 7, 82, jitter)
    for metric in (0, 1):
        _compare(oracle, "hex", xyz, cells, iters=2, nq=nq, grid_scale=grid_scale, extent=0, hex_metric=metric)


@pytest.mark.parametrize("k", [3, 6, 7, 13, 32])
@pytest.mark.parametrize("grid_scale", [0.1, 0.5, 2.0])
def test_hex_hubs(oracle, k, grid_scale):
    """rings of 6 to 64 hexes, 24 to 320 sub-tets: lists of several lane loads"""
    xyz, cells = _hex_fan(k, 6)
    for metric in (0, 1):
        _compare(oracle, "hex", xyz, cells, iters=2, grid_scale=grid_scale, extent=0, hex_metric=metric)


@pytest.mark.parametrize("nq", [2, 4, 6, 8])
@pytest.mark.parametrize("jitter,depth,extent,shift", [(0.3, 3, -1, 1000.0), (0.3, 7, -1, 0.0), (0.3, 3, 1, 0.0),
                                                       (0.9, 3, -1, 0.0), (0.0, 5, -1, 0.0)])
def test_tet_windows_that_the_planes_keep(oracle, nq, jitter, depth, extent, shift):
    """every candidate of a level: windows smaller than the planes' margins, far
    frames, inverted rings, regular ones; classes above the 4-wave form's 1,024"""
    xyz, cells = _cube("tet", 20, 83, jitter)
    xyz = (xyz.astype(np.float64) + shift).astype(np.float32)
    _compare(oracle, "tet", xyz, cells, iters=2, nq=nq, depth=depth, extent=extent)


@pytest.mark.parametrize("nq", [2, 4, 6, 8])
def test_tet_hub_in_a_batch(oracle, nq):
    """the one-wave search (a batch has no 4-wave form) on a ring of more
    elements than lanes, in windows of every size"""
    from volumesurfacediscretemeshoptimization_amd import DMOBatch, DMOMeshTetFactory
    k = 40
    t = 2.0 * np.pi * np.arange(k) / k
    pts = np.array([[0.05, -0.03, 0.02]] + [[np.cos(a), np.sin(a), 0.0] for a in t] + [[0.0, 0.0, 1.0], [0.0, 0.0, -1.0]],
                   np.float32)
    cells = []
    for i in range(k):
        j = (i + 1) % k
        cells += [[0, 1 + i, 1 + j, k + 1], [0, 1 + j, 1 + i, k + 2]]
    cells = np.array(cells, np.int32)
    mesh = DMOMeshTetFactory.create(pts, cells)
    b = DMOBatch([mesh], persistent=False, nq=nq, depth=6, quality_guard=False)
    o = oracle.OracleMesh("tet", pts, cells)
    try:
        b.iterate(2)
        for _ in range(2):
            o.iterate(nq=nq, depth=6, grid_scale=0.5)
        assert np.array_equal(b.positions(0).view(np.uint32), o.positions().view(np.uint32))
    finally:
        b.close()
        mesh.close()


@pytest.mark.parametrize("nq", [4, 8])
@pytest.mark.parametrize("policy", ["immediate", "deferred"])
@pytest.mark.parametrize("jitter", [0.0, 0.02, 0.3, 0.49])
def test_hex_fallback_lists_on_4_waves(oracle, monkeypatch, nq, policy, jitter):
    """learned hexes with the largest offset as extent: the fallbacks' full
    searches take 4 waves per vertex"""
    from test_gpu_learned_oracle import oracle_learned
    from volumesurfacediscretemeshoptimization_amd import DMOHexClass, DMOMeshHexFactory
    monkeypatch.setattr(oracle, "OR_EXTENT_MIN", oracle.OR_EXTENT_MAX)
    full = oracle.OracleMesh.search_vertex
    monkeypatch.setattr(oracle.OracleMesh, "search_vertex", lambda self, v, pos: full(self, v, pos, nq=nq))
    for xyz, cells in (_cube("hex", 6, 84, jitter), _hex_fan(10, 7)):
        for metric in (0, 1):
            ref, fb = oracle_learned(oracle, "hex", xyz, cells, None, 2, 1, 0.03125, policy, 2, hex_metric=metric)
            m = DMOMeshHexFactory.create(xyz, cells)
            o = DMOHexClass(m, n_iter=2, nq=nq, extent_mode=0, fixed_boundary=True, hex_metric=metric, quality_guard=False)
            try:
                o.set_proposal(None, mode=2, depth=1, window_frac=0.03125, fallback=policy)
                for it in range(2):
                    o.iterate(1)
                    gp = m.positions(original_order=False)
                    bad = (gp.view(np.uint32) != ref[it].view(np.uint32)).any(axis=1)
                    assert not bad.any(), (metric, it, int(bad.sum()), np.nonzero(bad)[0][:5])
                assert o.stats()["fallbacks"] == fb
            finally:
                o.close()
                m.close()
