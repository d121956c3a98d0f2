"""Batches that step through the element kernel's colour launches (a node of
63 elements or more): several groups with different shot and step counts,
sources and receivers, against the FP64 oracle; one launch per colour takes
every group, and kernel timing counts it once."""
import numpy as np
import pytest

from oracle import pyoracle as po
from salvus_amd import sem
from tests import problems as pb
from tests.test_gpu_elem_parts import fan

pytestmark = pytest.mark.gpu

TOL_RUN = 1e-5   # receiver relative L2 over a run (the metric's accuracy bar)


@pytest.mark.parametrize("physics", [0, 1])
@pytest.mark.parametrize("order", [1, 4])
def test_stepped_colours(physics, order, monkeypatch):
    monkeypatch.setenv("SEM_TIME_KERNELS", "1")
    meshes, B, want, ncol = [], sem.Batch(), [], 0
    dt, f0 = 2e-5, 200.0
    for k, shots, nsteps in ((63, 3, 40), (70, 1, 25), (70, 2, 40)):
        cells, coords = fan(k)
        par = pb.vertex_material(2, physics, cells, coords, np.random.default_rng(k))
        M = sem.Mesh(2, order, physics, cells, coords, par)
        meshes.append(M)
        ncol = max(ncol, 1 + int(M.colours().max()))
        for i in range(shots):
            O = po.Sim(2, order, physics, cells, coords, par)
            loc = coords[cells[(7 * i) % k]].mean(0)
            direction = np.array([0.3, 1.0])[:O.c]
            O.add_source(loc, 1e3, f0, 0.0, direction)
            j = B.add_shot(M, nsteps, dt)
            B.add_source(j, loc, 1e3, f0, 0.0, direction)
            for r in (coords[cells[0]].mean(0), coords[cells[k // 2]].mean(0)):
                O.add_receiver(r)
                B.add_receiver(j, r)
            want.append(O.run(dt, nsteps))
    B.prepare(sem.PATH_FUSED, 2, 3)
    assert B.config()["groups"] == 3 and B.config()["tiled_groups"] == 0
    B.run(40)
    assert B.kernel_time()[1] == 40 * ncol
    for j, w in enumerate(want):
        assert np.linalg.norm(w) > 0 and pb.rel_l2(B.seismograms(j), w) < TOL_RUN
