"""Device memory of requests and batches: a server charges what its groups
allocate, admits what five arrays a shot allow whatever its kernels would
rather take, and a batch that only fits in the least memory is set up in it;
results are the same bit for bit."""
import ctypes as C
from contextlib import contextmanager

import numpy as np
import pytest

from salvus_amd import sem
from tests import problems as pb
from tests.test_zz_no_alloc import Hip, noalloc

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def free_memory(hip):
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.L.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@contextmanager
def only(left):
    """All of the device's memory but `left` bytes held meanwhile."""
    hip = Hip()
    hog = hip.alloc(free_memory(hip) - left)
    try:
        yield
    finally:
        hip.L.hipFree(hog)


def problem(dim, physics, order, nel, distorted):
    P = pb.make(dim, physics, nel, order=order, seed=6, distorted=distorted, nrec=2)
    M = sem.Mesh(dim, order, physics, P["cells"], P["coords"], P["par"])
    assert (M.ntiles == 0) == distorted
    s = P["src"]
    src = [dict(kind="force", loc=P["coords"][P["cells"][7 + 5 * k]].mean(0), amp=s["amp"], f0=s["f0"], t0=0.0, dir=s["dir"])
           for k in range(4)]
    P["recs"] = [P["coords"][P["cells"][e]].mean(0) for e in (8, 13, 18)]
    return P, M, src


def serve(P, M, src, nsteps, **kw):
    S = sem.Server(block_steps=8, **kw)
    ids = [S.submit(M, nsteps, P["dt"], [x], P["recs"]) for x in src]
    st = S.pump()
    S.drain()
    return st, [S.result(i) for i in ids]


@pytest.mark.parametrize("order,nel", [(1, 100), (2, 60)])
def test_charged_bytes(order, nel):
    """Deformed acoustic hexes of low order, whose partial results take eight and
    three arrays: the charge covers the device memory gone after admission, up
    to what the batch's tables, graph and allocation granularity take."""
    P, M, src = problem(3, 0, order, nel, True)
    serve(P, M, src, 8)  # what the mesh builds for itself is there
    S = sem.Server(block_steps=8)
    for x in src:
        S.submit(M, 40, P["dt"], [x], P["recs"])
    free = free_memory(Hip())
    st = S.pump()
    gone = free - free_memory(Hip())
    assert st["active"] == 4 and gone > 4 * 5 * 4 * M.G  # more than the five arrays a shot
    assert gone - 48 * MIB < st["bytes"] < gone + 48 * MIB
    S.close()


@pytest.mark.parametrize("dim,physics,order,nel,distorted", [
    (3, 0, 1, 20, True), (3, 0, 2, 12, True), (3, 1, 4, 6, True), (2, 1, 1, 30, True), (3, 1, 2, 13, False)])
def test_budget_of_five_arrays(dim, physics, order, nel, distorted):
    """Three requests under a budget of three times their waiting charge: all
    active at once, never past the budget, with the results of a server that
    has all the memory it wants."""
    P, M, src = problem(dim, physics, order, nel, distorted)
    free, want = serve(P, M, src[:3], 24)
    one = sem.Server(block_steps=8)
    need = one.request(one.submit(M, 24, P["dt"], [src[0]], P["recs"]))["bytes"]
    st, got = serve(P, M, src[:3], 24, hbm_budget=3 * need)
    assert free["bytes"] > 3 * need  # the route of choice takes more
    assert st["active"] == 3 and st["bytes"] <= 3 * need
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0
        np.testing.assert_array_equal(a, b)


def test_batch_in_the_least_memory():
    """48 shots of 100^3 deformed order-1 hexes with 1400 MiB of the device left:
    five arrays a shot (0.99 GB) fit, the twelve of partial results (2.37 GB) do
    not."""
    P, M, src = problem(3, 0, 1, 100, True)

    def run():
        B = sem.Batch()
        for k in range(48):
            B.add_shot(M, 12, P["dt"])
            s = src[k % 4]
            B.add_source(k, s["loc"], s["amp"], s["f0"], s["t0"], s["dir"])
        B.prepare(sem.PATH_FUSED, 32, 4)
        B.run(12)
        out = [B.get_field(k, "u") for k in (0, 47)]
        B.close()
        return out

    want = run()
    with only(1400 * MIB):
        got = run()
    for a, b in zip(got, want):
        assert np.abs(b).max() > 0
        np.testing.assert_array_equal(a, b)


def test_operator_keeps_nothing_that_is_missed():
    """The allocation-free operator keeps its partial results with a mesh while
    they are less than a thousandth of the free memory; without them it gives
    the same bits."""
    P = pb.make(3, 1, 16, seed=7)
    u = np.random.default_rng(1).normal(size=(3, (16 * 4 + 1) ** 3)).astype(np.float32)
    M = sem.Mesh(3, 4, 1, P["cells"], P["coords"], P["par"])
    want = noalloc(M, u, Hip())
    with only(4096 * MIB):
        M2 = sem.Mesh(3, 4, 1, P["cells"], P["coords"], P["par"])
        got = noalloc(M2, u, Hip())
    assert M2.device_bytes < M.device_bytes - 4 * 16 ** 3 * 125
    np.testing.assert_array_equal(got, want)


@contextmanager
def exactly(left):
    """As `only`, until no more than `left` bytes are free (once memory is held,
    the runtime gives out some 500 MiB more than it had called free)."""
    hip, hogs = Hip(), []
    try:
        while (n := free_memory(hip) - left) > 0 and len(hogs) < 20:
            hogs.append(hip.alloc(n))
        yield
    finally:
        for h in hogs:
            hip.L.hipFree(h)


def test_dirichlet_mask_without_memory():
    """A mask set where the device has no memory for a second gather map (72 MB
    here) gives what it gives otherwise; so does taking it off again."""
    P, M, src = problem(3, 0, 4, 52, True)
    rng = np.random.default_rng(3)
    u = rng.normal(size=(1, M.G))
    mask = (rng.random(M.G) < 0.3).astype(np.uint8)
    free = M.apply_stiffness(u)
    M.set_dirichlet(mask)
    want = M.apply_stiffness(u)
    assert np.abs(want[:, mask == 1]).max() == 0 < np.abs(free[:, mask == 1]).max()
    with exactly(32 * MIB):
        M.set_dirichlet(np.zeros_like(mask))
    np.testing.assert_array_equal(M.apply_stiffness(u), free)
    with exactly(32 * MIB):
        M.set_dirichlet(mask)
    np.testing.assert_array_equal(M.apply_stiffness(u), want)


def test_mesh_that_just_fits():
    """40^3 deformed elastic hexes take 0.68 GiB of device memory and 0.09 GiB for
    a while; with 0.70 GiB left the mesh is made, and its operator is the same."""
    P = pb.make(3, 1, 40, seed=2, distorted=True)
    args = (3, 4, 1, P["cells"], P["coords"], P["par"])
    u = np.random.default_rng(1).normal(size=(3, (40 * 4 + 1) ** 3))
    want = sem.Mesh(*args).apply_stiffness(u)
    with exactly(720 * MIB):
        M = sem.Mesh(*args)
    np.testing.assert_array_equal(M.apply_stiffness(u), want)


def test_prepared_again_with_memory():
    """A batch that could not be set up for want of memory takes its kernels of
    choice (2.37 GB here, of which five arrays a shot are 0.99) when there is
    memory again."""
    P, M, src = problem(3, 0, 1, 100, True)
    B = sem.Batch()
    for k in range(48):
        B.add_shot(M, 12, P["dt"])
    with exactly(256 * MIB):
        with pytest.raises(sem.SemError, match="memory"):
            B.prepare(sem.PATH_FUSED, 32, 4)
    before = free_memory(Hip())
    B.prepare(sem.PATH_FUSED, 32, 4)
    assert before - free_memory(Hip()) > 2 << 30
