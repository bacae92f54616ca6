"""The brick kernel (AUTO on small and ordinary order-1 grids) against the
per-cell gather kernel: RHS, steps, time control, stage maxima and positivity
counts, all bit for bit, on brick edges, remainders, one-cell grids, every
border condition, periodic wraps and bodies."""
import numpy as np
import pytest

from test_gpu_kernels import build, run_variant

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


@pytest.mark.parametrize("name,dim,n,bc,body", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("negative", [False, True])
def test_brick_equals_gather(mmf, name, dim, n, bc, body, negative):
    info = np.zeros((6, 5))
    info[:] = [1.0, 0.3, -0.1, 0.05 if dim == 3 else 0.0, 1.0]
    s, U = build(mmf, dim, list(n), bc, info, body, seed=len(name))
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
        first = s.compute_rhs()
        counts = s.positivity_counters()
        if negative:
            s.advance(1)
            out.append((first, counts, s.nonfinite_steps(), s.get_state()))
        else:
            out.append((first, counts, run_variant(mmf, s, U, kind)))
    (Ra, ea), (Rb, eb) = out[0][0], out[1][0]
    assert np.array_equal(Ra, Rb, equal_nan=True) and (ea == eb or (np.isnan(ea) and np.isnan(eb)))
    assert out[0][1] == out[1][1]
    if negative:
        assert out[0][1][1] > 0 and out[0][2] == out[1][2]
        assert np.array_equal(out[0][3], out[1][3], equal_nan=True)
        return
    a, b = out[0][2], out[1][2]
    assert np.array_equal(a[0], b[0]) and a[1] == b[1]
    assert np.array_equal(a[2], b[2]), "state after 3 steps"
    assert a[3] == b[3], "time control and stage maxima"
    assert a[4] == b[4], "positivity counts"


def test_brick_steps_against_the_oracle(mmf, orc):
    """64^2 and 20 x 18 x 12, reflecting and Dirichlet sides, four steps each."""
    for dim, n, bc in ((2, [64, 64], [1, 1, 1, 1, 0, 0]), (3, [20, 18, 12], [3, 0, 1, 2, 0, 1])):
        info = np.tile([1.0, 0.3, -0.1, 0.0, 1.0], (6, 1))
        s, U = build(mmf, dim, n, bc, info, None, seed=9)
        h = 2.0 / max(n)
        o = orc.Solver(orc.problem(orc.RADSOD, dim), 1, n, [-1.0, -1.0, -1.0], h, side_bc=bc, side_info=info)
        Uo, W, t = U.copy(), U.copy(), 0.0
        s.set_state(U)
        s.set_time(0.0, 10.0, 0.5)
        for k in range(4):
            dt, _ = o.rk3_step(Uo, W, 0.5, t, 10.0)
            t += dt
            s.advance(1)
            assert s.time()[:2] == (t, dt)
        assert np.array_equal(s.get_state(), Uo)
