"""The batch autotuner times the schedules that differ: waves_per_vertex selects
no kernel, so it is not tuned (a wave count chosen by time was chosen by
noise), and a schedule's log lines hold one measurement.  The flat searches'
two kernels, 4 vertices per wave and one, on the same classes."""
import json

import numpy as np
import pytest

from volumesurfacediscretemeshoptimization_amd import (DMOBatch, DMOMeshTetFactory, DMOMeshTriFactory, DMOTriFlatClass,
                                                       synth)

pytestmark = pytest.mark.gpu


def test_one_measurement_per_schedule(tmp_path):
    m = [DMOMeshTetFactory.create(*synth.tet_cube(6, seed=1)), DMOMeshTriFactory.create(*synth.tri_grid(20, seed=2))]
    b = DMOBatch(m, waves_per_vertex=4)
    log = tmp_path / "tune.jsonl"
    try:
        chosen = b.autotune(iters=2, log_path=str(log))
        lines = [json.loads(x) for x in log.read_text().splitlines()]
        for persistent in (1, 0):
            t = {(x["waves_per_vertex"], x["ms_per_iter"]) for x in lines
                 if x["stage"] == "schedule" and x["persistent"] == persistent}
            assert {w for w, _ in t} == {1, 2, 4} and len({ms for _, ms in t}) == 1, t
        assert chosen["waves_per_vertex"] == 1 and b.params()["waves_per_vertex"] == 1
    finally:
        b.close()
        for x in m:
            x.close()


def test_flat_four_per_wave_equals_one_per_wave(oracle):
    """classes of 4,096 vertices and more: the optimiser takes the kernel of 4
    vertices per wave, a persistent batch the one of a vertex per wave"""
    xyz, tris = synth.tri_grid(160, seed=44)
    one, four = (DMOMeshTriFactory.create(xyz, tris) for _ in range(2))
    assert np.diff(four.color_offsets("free")).max() >= 4096
    opt = DMOTriFlatClass(four, n_iter=2, fixed_boundary=True)
    b = DMOBatch([one], persistent=True)
    o = oracle.OracleMesh("tri", xyz, tris)
    try:
        for it in range(2):
            opt.doIteration()
            b.iterate(1)
            o.iterate()
            ref = o.positions().view(np.uint32)
            assert np.array_equal(b.positions(0).view(np.uint32), ref), it
            assert np.array_equal(four.positions(original_order=False).view(np.uint32), ref), it
    finally:
        opt.close()
        b.close()
        one.close()
        four.close()
