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
