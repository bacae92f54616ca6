"""The brick kernels (AUTO on small and ordinary order-1 grids and on order-2
grids without a body) against the per-cell gather kernel: RHS, steps, time
control, stage maxima and positivity counts, all bit for bit, on brick edges,
remainders, one-cell grids, every border condition, periodic wraps and
bodies."""
import numpy as np
import pytest

from test_gpu_kernels import build

pytestmark = pytest.mark.gpu

CASES = [
    ("3d one cell", 3, (1, 1, 1), [0, 1, 2, 3, 0, 1], None),
    ("3d one brick", 3, (8, 8, 4), [3, 0, 1, 2, 0, 3], None),
    ("3d one past a brick", 3, (9, 9, 5), [1, 1, 0, 3, 2, 0], None),
    ("3d thin, wraps inside a brick", 3, (3, 17, 2), [4, 4, 1, 0, 4, 4], None),
    ("3d periodic, full bricks", 3, (16, 8, 4), [4] * 6, None),
    ("3d ragged", 3, (70, 13, 37), [0, 1, 2, 0, 1, 0], None),
    ("3d ragged periodic", 3, (33, 20, 11), [4, 4, 4, 4, 0, 2], None),
    ("3d box", 3, (40, 24, 20), [3, 0, 1, 1, 0, 2], {"boxes": [[-0.4, -0.3, -0.5, 0.1, 0.35, 0.2]]}),
    ("3d body across the wrap", 3, (130, 20, 24), [4, 4, 4, 4, 0, 3],
     {"boxes": [[0.9, -0.75, -0.9, 1.0, -0.68, -0.8]]}),
    ("3d body on the borders", 3, (20, 18, 12), [3, 1, 0, 3, 2, 3], {"spheres": [[-1.0, -1.0, -1.0, 0.6]]}),
    ("2d one cell", 2, (1, 1), [3, 0, 1, 2], None),
    ("2d 8 x 8 bricks", 2, (9, 8), [4, 4, 1, 3], None),
    ("2d wrap inside a brick", 2, (5, 17), [4, 4, 4, 4], None),
    ("2d reflecting", 2, (77, 50), [1, 1, 2, 1], None),
    ("2d 16 x 16 bricks, ragged", 2, (300, 261), [3, 0, 1, 2], None),
    ("2d 16 x 16 bricks, periodic", 2, (272, 257), [4, 4, 4, 4], None),
    ("2d cylinder", 2, (50, 44), [3, 0, 1, 0], {"spheres": [[0.1, -0.05, -1.0, 0.3]]}),
    ("2d cylinder, 16 x 16 bricks", 2, (260, 270), [3, 0, 0, 0], {"spheres": [[0.1, -0.05, -1.0, 0.3]]}),
]


O2_CASES = [
    ("3d o2 one cell", 3, (1, 1, 1), [0, 1, 2, 3, 0, 1]),
    ("3d o2 one brick", 3, (8, 8, 4), [3, 0, 1, 2, 0, 3]),
    ("3d o2 one past a brick", 3, (9, 9, 5), [1, 1, 0, 3, 2, 0]),
    ("3d o2 two cells per axis, periodic", 3, (2, 2, 2), [4] * 6),
    ("3d o2 thin, wraps inside a brick", 3, (3, 17, 2), [4, 4, 1, 0, 4, 4]),
    ("3d o2 full bricks, periodic", 3, (16, 8, 12), [4] * 6),
    ("3d o2 ragged", 3, (70, 13, 37), [0, 1, 2, 0, 1, 3]),
    # 2D: one-wave bricks above 2^14 cells
    ("2d o2 one past a brick", 2, (129, 137), [1, 2, 0, 3]),
    ("2d o2 two columns, periodic", 2, (2, 8201), [4] * 4),
    ("2d o2 one row", 2, (16385, 1), [0, 2, 1, 3]),
    ("2d o2 large", 2, (530, 510), [3, 0, 4, 4]),
]


@pytest.mark.parametrize("name,dim,n,bc", O2_CASES, ids=[c[0] for c in O2_CASES])
@pytest.mark.parametrize("negative", [False, True])
def test_brick_order2_equals_gather(mmf, name, dim, n, bc, negative):
    check(mmf, name, dim, n, bc, None, negative, 2)


@pytest.mark.parametrize("name,dim,n,bc,body", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("negative", [False, True])
def test_brick_equals_gather(mmf, name, dim, n, bc, body, negative):
    check(mmf, name, dim, n, bc, body, negative, 1)


def check(mmf, name, dim, n, bc, body, negative, order):
    info = np.zeros((6, 5))
    info[:] = [1.0, 0.3, -0.1, 0.05 if dim == 3 else 0.0, 1.0]
    s, U = build(mmf, dim, list(n), bc, info, body, order=order, seed=len(name))
    if negative:  # density and energy negative: real sound speed, counted sides
        k = np.random.default_rng(3).integers(0, len(U), max(1, len(U) // 50))
        U = U.copy()
        U[k, 0] *= -1.0
        U[k, 4] *= -1.0
    out = []
    for kind in (mmf.KERNEL_GATHER, mmf.KERNEL_AUTO):
        s.set_time(0.0, 10.0, 0.5)
        s.reset_positivity_counters()
        s.set_kernel(kind)
        s.set_state(U)
        rhs, eig = s.compute_rhs()
        counts = [s.positivity_counters()]
        s.advance(1 if negative else 3)
        try:
            t, dt, step, stages = s.time()
            time = (t, dt, step, tuple(stages))
        except mmf.MMFError:  # the flow itself left the positive states, with either kernel
            time = s.nonfinite_steps()
        counts.append(s.positivity_counters())
        out.append((rhs, eig, s.get_state(), time, counts))
    a, b = out
    assert np.array_equal(a[0], b[0], equal_nan=True), "rhs"
    assert a[1] == b[1] or (np.isnan(a[1]) and np.isnan(b[1])), "maximum eigenvalue"
    assert np.array_equal(a[2], b[2], equal_nan=True), "state after the steps"
    assert a[3] == b[3], "time control and stage maxima"
    if negative:
        assert a[4][0][1] > 0
        assert a[4][0] == b[4][0], "positivity counts"
    else:
        assert a[4] == b[4], "positivity counts"


STEP_CASES = [
    ("one cell", (1, 1), [3, 0, 1, 2]),
    ("two cells per axis, periodic", (2, 2), [4] * 4),
    ("wraps several times", (2, 3), [4, 4, 4, 4]),
    ("one tile", (10, 10), [1, 3, 2, 0]),
    ("one past a tile", (11, 21), [4, 4, 3, 1]),
    ("borders in the last ring", (12, 13), [0, 1, 3, 2]),
    ("one row", (129, 1), [0, 2, 1, 3]),
    ("largest, ragged", (257, 255), [3, 0, 1, 2]),
    ("periodic", (64, 50), [4] * 4),
]


@pytest.mark.parametrize("name,n,bc", STEP_CASES, ids=[c[0] for c in STEP_CASES])
@pytest.mark.parametrize("negative", [False, True])
def test_steps_in_one_launch_equal_gather(mmf, name, n, bc, negative):
    """Pairs of steps, each one launch on a small 2D grid, and a final time
    reached by the first step of a pair (the other one then only moves the
    state back)."""
    info = np.tile([1.0, 0.3, -0.1, 0.0, 1.0], (6, 1))
    s, U = build(mmf, 2, list(n), bc, info, None, order=1, seed=len(name))
    if negative:
        k = np.random.default_rng(3).integers(0, len(U), max(1, len(U) // 50))
        U = U.copy()
        U[k, 0] *= -1.0
        U[k, 4] *= -1.0
    s.set_kernel(mmf.KERNEL_GATHER)
    s.set_state(U)
    s.set_time(0.0, 10.0, 0.5)
    s.advance(1)
    try:
        ends = [10.0] if negative else [10.0, 2.5 * s.time()[1]]
    except mmf.MMFError:
        ends = [10.0]
    for end in ends:
        out = []
        for kind in (mmf.KERNEL_GATHER, mmf.KERNEL_AUTO):
            s.set_kernel(kind)
            s.set_state(U)
            s.set_time(0.0, end, 0.5)
            s.reset_positivity_counters()
            s.advance(2 if negative else 4)
            try:
                t, dt, step, stages = s.time()
                time = (t, dt, step, tuple(stages))
            except mmf.MMFError:
                time = s.nonfinite_steps()
            out.append((s.get_state(), time, s.positivity_counters()))
        a, b = out
        assert np.array_equal(a[0], b[0], equal_nan=True), "state"
        assert a[1] == b[1], "time control and stage maxima"
        assert a[2] == b[2], "positivity counts"


def test_brick_steps_against_the_oracle(mmf, orc):
    """64^2 and 20 x 18 x 12, reflecting and Dirichlet sides, orders 1 and 2, four steps each."""
    for dim, n, bc, order in ((2, [64, 64], [1, 1, 1, 1, 0, 0], 1), (3, [20, 18, 12], [3, 0, 1, 2, 0, 1], 1),
                              (2, [60, 52], [3, 1, 4, 4, 0, 0], 2), (3, [20, 18, 12], [3, 0, 1, 2, 0, 1], 2)):
        info = np.tile([1.0, 0.3, -0.1, 0.0, 1.0], (6, 1))
        s, U = build(mmf, dim, n, bc, info, None, order=order, seed=9)
        h = 2.0 / max(n)
        o = orc.Solver(orc.problem(orc.RADSOD, dim), order, n, [-1.0, -1.0, -1.0], h, side_bc=bc, side_info=info)
        Uo, W, t = U.copy(), U.copy(), 0.0
        s.set_state(U)
        s.set_time(0.0, 10.0, 0.5)
        for k in range(4):
            dt, _ = o.rk3_step(Uo, W, 0.5, t, 10.0)
            t += dt
            s.advance(1)
            assert s.time()[:2] == (t, dt)
        assert np.array_equal(s.get_state(), Uo)
