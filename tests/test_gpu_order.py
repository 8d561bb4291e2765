"""Loads and solutions between the caller's DOF order and the internal one, on
either side of the size from which the device reorders them (16,384 nodes):
exact copies, so a unit load at each end of the mesh and the solution read
twice compare bitwise with the reordering done here from node_perm."""

import threading

import numpy as np
import pytest

from bfm_amd import device as D
from bfm_amd import meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(8, 3), (127, 127), (128, 127), (255, 64)])   # 36, 16384, 16512, 16640 nodes
def test_given_loads_and_solutions(nx, ny):
    m = meshgen.beam(nx, ny, kind=4, jitter=0.2, seed=2)
    s = D.beam_system(m)
    b = s.get_rhs()                                # the assembled load in the caller's order
    u, st = s.solve(precond=D.PRECOND_AMG, rtol=1e-8)
    assert np.array_equal(u, s.get_u())
    u2, st2 = s.solve(b=b, precond=D.PRECOND_AMG, rtol=1e-8)   # the same load handed in
    assert st2["iterations"] == st["iterations"] and np.array_equal(u, u2)
    A = s.get_csr_scipy()
    assert np.linalg.norm(b - A @ u) <= 1.1e-8 * np.linalg.norm(b)
    rng = np.random.default_rng(0)
    b3 = rng.standard_normal(b.size) * np.abs(b).max()
    b3.reshape(-1, 2)[m.node_sets["left"]] = 0
    u3, _ = s.solve(b=b3, precond=D.PRECOND_AMG, rtol=1e-8)
    assert np.linalg.norm(b3 - A @ u3) <= 1.1e-8 * np.linalg.norm(b3)


def test_a_thread_leaves_its_pinned_buffer_to_the_next():
    """Below 16,384 nodes a load and a solution go through a pinned buffer of the calling thread (256 KB here). Sixty
    threads one after another use one of them, not sixty: the process maps no more device memory than after the first
    few."""
    s = D.beam_system(meshgen.beam(127, 120, kind=4, jitter=0.2, seed=2))
    small = D.beam_system(meshgen.beam(8, 3, kind=4))
    b, b_small = s.get_rhs(), small.get_rhs()
    want, _ = s.solve(b=b, precond=D.PRECOND_AMG, rtol=1e-6)
    want_small, _ = small.solve(b=b_small, rtol=1e-6)
    wrong = []

    def mapped():
        with open("/proc/self/maps") as f:
            return sum("/dev/dri/" in line or "/dev/kfd" in line for line in f)

    def work(k):
        u, _ = s.solve(b=b, precond=D.PRECOND_AMG, rtol=1e-6)
        v, _ = small.solve(b=b_small, rtol=1e-6)
        if not (np.array_equal(u, want) and np.array_equal(s.get_u(), want) and np.array_equal(v, want_small)):
            wrong.append(k)

    counts = []
    for k in range(60):
        t = threading.Thread(target=work, args=(k,))
        t.start()
        t.join()
        counts.append(mapped())
    print(f"mapped: {counts[4]} after 5 threads, {counts[-1]} after {len(counts)}")
    assert not wrong
    assert counts[4] > 0 and counts[-1] <= counts[4] + 4


def test_batches_on_two_threads_share_a_large_system():
    """Both batches read the solution of the same system, whose permutation goes to the device at the first read."""
    s = D.beam_system(meshgen.beam(255, 64, kind=3, jitter=0.2, seed=2))
    batches = [D.Batch([s]) for _ in range(2)]
    got = [None, None]

    def work(k):
        batches[k].solve(rtol=1e-6)
        got[k] = batches[k].get_u(0)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert np.array_equal(got[0], got[1])
    A, b = s.get_csr_scipy(), s.get_rhs()
    assert np.linalg.norm(b - A @ got[0]) <= 1.1e-6 * np.linalg.norm(b)
