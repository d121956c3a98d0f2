"""Colour launches of the tile kernel (large 3-D batches; SEM_TILE_OCCUPANCY for
acoustic meshes of any size, in both occupancy variants) against the launch
over all tiles: bit for bit, on boxes of one tile, of one tile and one more
element along an axis, and ragged ones, with several shots, Dirichlet nodes set
after prepare, and coupled shots."""
import numpy as np
import pytest

from salvus_amd import meshgen, sem
from tests import problems as pb
from tests import test_gpu_coupled as coupled

pytestmark = pytest.mark.gpu


def fields(M, P, shots, nsteps, mask, which):
    dim = P["coords"].shape[1]
    B = sem.Batch()
    for j in range(shots):
        B.add_shot(M, nsteps, 2e-5)
        B.add_source(j, P["coords"][P["cells"][j % len(P["cells"])]].mean(0), 1e3, 200.0, 0.0, np.arange(1.0, M.c + 1))
        for e in (0, len(P["cells"]) // 2, len(P["cells"]) - 1):
            B.add_receiver(j, P["coords"][P["cells"][e]].mean(0) + 0.4)
        if j in which:
            B.set_field(j, "u", np.random.default_rng(j).normal(size=(M.c, M.G)))
    B.prepare(sem.PATH_FUSED, 1, 4)
    assert B.config()["tiled_groups"] == B.config()["groups"]
    if mask is not None:
        M.set_dirichlet(mask)
    B.run(nsteps)
    launches = B.kernel_time()[1]
    if mask is not None:
        M.set_dirichlet(np.zeros(M.G, bool))
    return launches, [x for j in which for x in (B.get_field(j, "u"), B.get_field(j, "v"), B.seismograms(j))]


@pytest.mark.parametrize("mode", ["normal", "high"])
@pytest.mark.parametrize("order", [2, 4])
@pytest.mark.parametrize("box", [(16, 8), (17, 8), (33, 17), (4, 4, 2), (5, 2, 2), (4, 3, 3), (9, 5, 3)])
def test_acoustic_modes(box, order, mode, monkeypatch):
    dim = len(box)
    cells, coords = (meshgen.box_quad if dim == 2 else meshgen.box_hex)(*box, *[10.0 * n for n in box])
    P = dict(cells=cells, coords=coords)
    M = sem.Mesh(dim, order, 0, cells, coords, pb.vertex_material(dim, 0, cells, coords, np.random.default_rng(1)))
    mask = np.random.default_rng(2).random(M.G) < 0.1
    monkeypatch.setenv("SEM_TIME_KERNELS", "1")
    for m in (None, mask):
        n0, want = fields(M, P, 5, 9, m, range(5))
        with monkeypatch.context() as mp:
            mp.setenv("SEM_TILE_OCCUPANCY", mode)
            n1, got = fields(M, P, 5, 9, m, range(5))
        assert n0 == 9 and n1 == 9 * np.prod([min(2, -(-n // t)) for n, t in zip(box, M.tile_shape)])
        for a, b in zip(got, want):
            np.testing.assert_array_equal(a, b)
    u = np.random.default_rng(3).normal(size=(1, M.G))
    want = M.apply_stiffness(u)
    monkeypatch.setenv("SEM_TILE_OCCUPANCY", mode)
    np.testing.assert_array_equal(M.apply_stiffness(u), want)


@pytest.mark.parametrize("box,shots", [((33, 31, 32), 18)])
def test_elastic_large_batch(box, shots, monkeypatch):
    """2304 tiles of order 5 (one workgroup a CU), 18 shots: colour launches; the
    same shots alone: one launch and the shared nodes."""
    cells, coords = meshgen.box_hex(*box, *[10.0 * n for n in box])
    P = dict(cells=cells, coords=coords)
    M = sem.Mesh(3, 5, 1, cells, coords, pb.vertex_material(3, 1, cells, coords, np.random.default_rng(4)))
    mask = np.random.default_rng(5).random(M.G) < 0.05
    monkeypatch.setenv("SEM_TIME_KERNELS", "1")
    n8, got = fields(M, P, shots, 5, mask, (0, 1))
    n1, want = fields(M, P, 2, 5, mask, (0, 1))
    assert n8 == 8 * 5 and n1 == 5
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("mode", ["normal", "high"])
def test_coupled_fluid(mode, monkeypatch):
    """The external load starts a node's sum in its first colour: the coupled run's
    own test (FP64 oracle) with the fluid in colour launches."""
    monkeypatch.setenv("SEM_TILE_OCCUPANCY", mode)
    coupled.test_coupled_run(sem.PATH_FUSED, "straight", False, "f", False)


@pytest.mark.parametrize("half", [False, True])
def test_split_mesh_keeps_partial_results(half, monkeypatch):
    """A box cut along a tile boundary (wholly, or up to its middle) is tiled, but
    its tiles do not share all nodes of that face: no colour launches."""
    box, at = (8, 8, 4), 4
    cells, coords = meshgen.box_hex(*box, *[10.0 * n for n in box])
    par = pb.vertex_material(3, 0, cells, coords, np.random.default_rng(1))
    right = coords[cells].mean(1)[:, 0] > 10.0 * at
    cut = np.flatnonzero((coords[:, 0] == 10.0 * at) & ((coords[:, 1] < 35.0) | (not half)))
    twin = np.arange(len(coords))
    twin[cut] = len(coords) + np.arange(len(cut))
    cells = np.where(right[:, None], twin[cells], cells)
    coords = np.vstack([coords, coords[cut]])
    M = sem.Mesh(3, 4, 0, cells, coords, par)
    assert M.ntiles == 2 * 2 * 2 and M.tile_shape == (4, 4, 2)
    P = dict(cells=cells, coords=coords)
    monkeypatch.setenv("SEM_TIME_KERNELS", "1")
    n0, want = fields(M, P, 2, 9, None, range(2))
    monkeypatch.setenv("SEM_TILE_OCCUPANCY", "normal")
    n1, got = fields(M, P, 2, 9, None, range(2))
    assert n0 == 9 and n1 == 9
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)
