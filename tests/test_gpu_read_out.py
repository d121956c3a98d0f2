"""Field read-out: several threads reading shots of one batch at once each get
their own values, and the first read allocates nothing on the device."""
import threading

import numpy as np
import pytest

from salvus_amd import sem
from tests import problems as pb
from tests.test_gpu_memory import free_memory
from tests.test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


def batch(nel, shots, dim=3, distorted=False):
    P = pb.make(dim, 1, nel, seed=8, distorted=distorted)
    M = sem.Mesh(dim, 4, 1, P["cells"], P["coords"], P["par"])
    B = sem.Batch()
    u = []
    for j in range(shots):
        B.add_shot(M, 10, P["dt"])
        u.append(np.random.default_rng(j).normal(size=(M.c, M.G)).astype(np.float32).astype(np.float64))
        for which in ("u", "v"):
            B.set_field(j, which, u[j])
    B.prepare(sem.PATH_FUSED, 1, shots)
    return M, B, u


@pytest.mark.parametrize("distorted", [False, True])
def test_threads_read_their_own_shot(distorted):
    M, B, u = batch(12, 4, distorted=distorted)
    wrong = []

    def read(j):
        for _ in range(60):
            if not np.array_equal(B.get_field(j, "u"), u[j]):
                wrong.append(j)

    threads = [threading.Thread(target=read, args=(j,)) for j in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


def test_first_read_allocates_nothing():
    M, B, u = batch(30, 1)
    free = free_memory(Hip())
    np.testing.assert_array_equal(B.get_field(0, "u"), u[0])
    assert free_memory(Hip()) == free


@pytest.mark.parametrize("path", [sem.PATH_FUSED, sem.PATH_PLAIN])
@pytest.mark.parametrize("dim,nel,distorted", [(2, 30, False), (2, 90, False), (2, 90, True), (3, 12, False),
                                               (3, 21, True)])
def test_in_one_or_several_pieces(path, dim, nel, distorted):
    """Fields that fit the space for them, that take several pieces and that go
    through the partial results; the steps that follow are those of a batch
    that was never read."""
    M, B, u = batch(nel, 2, dim, distorted)
    M2, B2, _ = batch(nel, 2, dim, distorted)
    if path == sem.PATH_PLAIN:
        for b in (B, B2):
            b.close()
        P = pb.make(dim, 1, nel, seed=8, distorted=distorted)
        B, B2 = sem.Batch(), sem.Batch()
        for b in (B, B2):
            for j in range(2):
                b.add_shot(M, 10, P["dt"])
                for which in ("u", "v"):
                    b.set_field(j, which, u[j])
            b.prepare(path, 1, 1)
    for j in range(2):
        np.testing.assert_array_equal(B.get_field(j, "u"), u[j])
        np.testing.assert_array_equal(B.get_field(j, "v"), u[j])
    for _ in range(3):
        B.run(2)
        got = [B.get_field(j, "u") for j in range(2)]
    B2.run(6)
    for j in range(2):
        np.testing.assert_array_equal(got[j], B2.get_field(j, "u"))


@pytest.mark.parametrize("distorted", [False, True])
def test_read_while_stepping(distorted, monkeypatch):
    """A thread that reads while another one steps gets the field after some
    whole block of steps."""
    monkeypatch.setenv("SEM_GRAPH_STEPS", "2")
    P = pb.make(3, 1, 24, seed=8, distorted=distorted)
    M = sem.Mesh(3, 4, 1, P["cells"], P["coords"], P["par"])
    u0 = np.random.default_rng(1).normal(size=(M.c, M.G)).astype(np.float32).astype(np.float64)
    steps = 30

    def start():
        b = sem.Batch()
        b.add_shot(M, steps, P["dt"])
        b.set_field(0, "u", u0)
        b.prepare(sem.PATH_FUSED, 1, 1)
        return b

    B, R = start(), start()
    seen = [R.get_field(0, "u")]
    for _ in range(steps // 2):
        R.run(2)
        seen.append(R.get_field(0, "u"))
    t = threading.Thread(target=B.run, args=(steps,))
    t.start()
    got = [B.get_field(0, "u") for _ in range(8)]
    t.join()
    got.append(B.get_field(0, "u"))
    at = [[k for k, s in enumerate(seen) if np.array_equal(g, s)] for g in got]
    assert all(at) and at[-1] == [steps // 2]
