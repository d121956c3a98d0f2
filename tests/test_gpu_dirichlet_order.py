"""Dirichlet nodes set on a mesh whose batches are already prepared, or whose
requests are active in a server, act on every node from the next run on, as a
mask set beforehand does: bit for bit, on the tile kernel (nodes inside a tile
and nodes that tiles share) and on the element kernel."""
import numpy as np
import pytest

from salvus_amd import sem
from tests import problems as pb

pytestmark = pytest.mark.gpu

CASES = [(2, 0, False), (2, 1, False), (3, 0, False), (3, 1, False), (2, 1, True), (3, 0, True)]


def problem(dim, physics, distorted):
    P = pb.make(dim, physics, 6 if dim == 3 else 20, seed=9, distorted=distorted, nsteps=24)
    M = sem.Mesh(dim, 4, physics, P["cells"], P["coords"], P["par"])
    assert (M.ntiles == 0) == distorted
    xyz = M.node_coords()
    mask = (np.abs(xyz[:, 0]) < 1e-9) | (np.abs(xyz[:, 1] - P["L"]) < 1e-9) | (np.random.default_rng(1).random(M.G) < 0.1)
    return P, M, mask


def batch(P, M):
    B = sem.Batch()
    B.add_shot(M, 24, P["dt"])
    s = P["src"]
    B.add_source(0, s["loc"], s["amp"], s["f0"], 0.0, s["dir"])
    for r in P["recs"]:
        B.add_receiver(0, r)
    B.set_field(0, "u", np.random.default_rng(2).normal(size=(M.c, M.G)) * 1e-9)
    B.prepare(sem.PATH_FUSED, 1, 1)
    return B


@pytest.mark.parametrize("dim,physics,distorted", CASES)
def test_mask_after_prepare(dim, physics, distorted):
    P, M, mask = problem(dim, physics, distorted)
    free, late = batch(P, M), batch(P, M)
    free.run(24)
    M.set_dirichlet(mask)
    late.run(24)
    early = batch(P, M)
    early.run(24)
    np.testing.assert_array_equal(late.get_field(0, "u"), early.get_field(0, "u"))
    np.testing.assert_array_equal(late.seismograms(0), early.seismograms(0))
    assert not np.array_equal(free.get_field(0, "u"), early.get_field(0, "u"))
    M.set_dirichlet(np.zeros(M.G, bool))  # and taken off again
    again = batch(P, M)
    M.set_dirichlet(mask)
    M.set_dirichlet(np.zeros(M.G, bool))
    again.run(24)
    np.testing.assert_array_equal(again.get_field(0, "u"), free.get_field(0, "u"))


@pytest.mark.parametrize("dim,physics,distorted", CASES)
def test_mask_while_a_request_is_active(dim, physics, distorted):
    P, M, mask = problem(dim, physics, distorted)
    s = P["src"]
    src = dict(kind="force", loc=s["loc"], amp=s["amp"], f0=s["f0"], t0=0.0, dir=s["dir"])
    S = sem.Server(block_steps=8)
    rid = S.submit(M, 24, P["dt"], [src], P["recs"])
    S.pump()
    M.set_dirichlet(mask)
    S.drain()
    M.set_dirichlet(np.zeros(M.G, bool))
    out = []
    for masked in (True, False):
        B = sem.Batch()
        B.add_shot(M, 24, P["dt"])
        B.add_source(0, s["loc"], s["amp"], s["f0"], 0.0, s["dir"])
        for r in P["recs"]:
            B.add_receiver(0, r)
        B.prepare(sem.PATH_FUSED, 1, 1)
        B.run(8)
        if masked:
            M.set_dirichlet(mask)
        B.run(16)
        M.set_dirichlet(np.zeros(M.G, bool))
        out.append(B.seismograms(0))
    np.testing.assert_array_equal(S.result(rid), out[0])
    assert not np.array_equal(out[0], out[1])
