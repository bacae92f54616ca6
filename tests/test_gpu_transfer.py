"""States and residuals across the host link: sizes on both sides of where the
rows are formed on the host or the device and where the copy goes through
pinned chunks, several threads at once, and the chunks released and made anew."""
import threading

import numpy as np
import pytest

from minimmerflow_amd import meshes

pytestmark = pytest.mark.gpu


def rows(N, seed=0):
    r = np.random.default_rng(seed + N)
    U = r.standard_normal((N, 5))
    U[:, 0] = 1.0 + 0.1 * r.uniform(size=N)
    U[:, 4] = 3.0 + r.uniform(size=N)
    return U


# 5120 and 12288 cells: host or device rows; 52,428.8 cells: 2 MB, the pinned
# chunks of 1 MB, a ring of twelve of them
SIZES = [1, 63, 64, 65, 5119, 5120, 12287, 12288, 52428, 52429, 78643, 78644, 314573, 700001]


@pytest.mark.parametrize("N", SIZES)
def test_states_come_back(mmf, N):
    U, V = rows(N), rows(N, 1)
    s = mmf.Solver(2, [N, 1], [0.0] * 3, 0.01, [0] * 4)
    b = mmf.Batch([mmf.grid_desc(2, [N, 1], [0.0] * 3, 0.01, [0] * 4), mmf.grid_desc(2, [1, N], [0.0] * 3, 0.01, [0] * 4)])
    s.set_state(U)
    b.set_state(0, U)
    b.set_state(1, V)
    assert np.array_equal(s.get_state(), U)
    assert np.array_equal(b.get_state(0), U) and np.array_equal(b.get_state(1), V)
    s.set_state(V)
    b.set_state(0, V)
    assert np.array_equal(s.get_state(), V) and np.array_equal(b.get_state(0), V)
    s.close()
    b.close()


@pytest.mark.parametrize("n", [(1, 2), (70, 73), (64, 80), (111, 110), (128, 96), (300, 200)])
def test_face_list_states_come_back(mmf, n):
    fm = meshes.cartesian(2, list(n), [0.0] * 3, 0.25, [0] * 4)
    g = mmf.Mesh(fm)
    for seed in (0, 1):
        U = rows(fm.ncells, seed)
        g.set_state(U)
        assert np.array_equal(g.get_state(), U)
        s = mmf.Solver(2, list(n), [0.0] * 3, 0.25, [0] * 4)
        s.set_state(U)
        assert np.array_equal(g.compute_rhs()[0], s.compute_rhs()[0], equal_nan=True)  # some pressures are negative
        s.close()
    g.close()


def test_threads_read_at_once(mmf):
    """Only one of them holds the chunks; the others' copies are plain."""
    N, count = 400003, 4
    solvers = [mmf.Solver(2, [N, 1], [0.0] * 3, 0.01, [0] * 4) for _ in range(count)]
    states = [rows(N, k) for k in range(count)]
    bad = []

    def work(k):
        s, U = solvers[k], states[k]
        s.set_state(U)
        for i in range(6):
            if not np.array_equal(s.get_state(), U):
                bad.append((k, i))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(count)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in solvers:
        s.close()
    assert not bad


def test_chunks_after_the_last_object(mmf):
    """The chunks go with the last object and come back with the next large copy,
    also while another thread's object goes."""
    N = 300007
    U = rows(N)
    for _ in range(4):
        s = mmf.Solver(2, [N, 1], [0.0] * 3, 0.01, [0] * 4)
        s.set_state(U)
        other = mmf.Solver(2, [8, 8], [0.0] * 3, 0.01, [0] * 4)
        t = threading.Thread(target=other.close)
        t.start()
        assert np.array_equal(s.get_state(), U)
        t.join()
        s.close()
