"""Which stage kernel runs: mmf_get_kernel names it, mmf_set_kernel takes that
name, and the bricks asked for by name equal the per-cell gather kernel on
every case of the brick tests, whatever AUTO picks there."""
import types

import numpy as np
import pytest

from test_gpu_brick import CASES, O2_CASES, check
from test_gpu_kernels import build

pytestmark = pytest.mark.gpu

INFO = np.tile([1.0, 0.3, -0.1, 0.0, 1.0], (6, 1))


@pytest.mark.parametrize("negative", [False, True])
@pytest.mark.parametrize("name,dim,n,bc,body", CASES + [c + (None,) for c in O2_CASES if c[1] == 3],
                         ids=[c[0] for c in CASES + O2_CASES if c in CASES or c[1] == 3])
def test_bricks_by_name_equal_gather(mmf, name, dim, n, bc, body, negative):
    order = 2 if " o2 " in name else 1
    s, _ = build(mmf, dim, list(n), bc, INFO, body, order=order, seed=1)
    s.set_kernel(mmf.KERNEL_BRICK)
    assert s.kernel()[0] == mmf.KERNEL_BRICK
    s.close()
    named = types.SimpleNamespace(**dict(vars(mmf), KERNEL_AUTO=mmf.KERNEL_BRICK))
    check(named, name, dim, n, bc, body, negative, order)


AUTO_KINDS = [
    (2, (64, 64), 1, "BRICK"),
    (2, (300, 260), 1, "BRICK"),
    (2, (1000, 600), 1, "BRICK"),
    (3, (32, 32, 32), 1, "BRICK"),
    (3, (100, 90, 84), 1, "BRICK"),
    (3, (256, 128, 64), 1, "MARCH"),
    (2, (100, 100), 2, "TILE"),
    (2, (600, 500), 2, "TILE"),
    (2, ((1 << 14) - 1, 1 << 14), 2, "TILE"),
    (2, (1 << 14, 1 << 14), 2, "MARCH"),  # beyond the bricks' cells
    # a few cells across: not to bricks of mostly padding, unless they are few
    (2, (7680, 1), 1, "BRICK"),
    (2, (60000, 1), 1, "GATHER"),
    (2, (1, 200000), 1, "GATHER"),
    (2, (500000, 2), 1, "MARCH"),
    (2, (2, 500000), 1, "GATHER"),
    (2, (8, 100000), 1, "BRICK"),
    (3, (1000, 1, 1), 1, "BRICK"),
    (3, (60000, 1, 1), 1, "GATHER"),
    (3, (1, 1, 400000), 1, "GATHER"),
    (3, (60000, 4, 4), 1, "BRICK"),
    (3, (1100, 1, 1100), 1, "GATHER"),
    (3, (1100, 1100, 1), 1, "MARCH"),
    (3, (550, 4, 550), 1, "MARCH"),
    (3, (4, 550, 550), 1, "BRICK"),
    (2, (200000, 1), 2, "GATHER"),
    (2, (500000, 4), 2, "MARCH"),
    (2, (100000, 4), 2, "TILE"),
    (3, (60000, 1, 1), 2, "GATHER"),
    (3, (300, 3, 300), 2, "BRICK"),
    (3, (800, 2, 800), 2, "GATHER"),
    (3, (1100, 1100, 1), 2, "MARCH"),
    (3, (32, 32, 32), 2, "BRICK"),
    (3, (144, 144, 144), 2, "BRICK"),
]


@pytest.mark.parametrize("dim,n,order,kind", AUTO_KINDS)
def test_the_kind_in_use_is_named_and_taken(mmf, dim, n, order, kind):
    s = mmf.Solver(dim, list(n), [0.0] * 3, 0.01, [0] * 6, None, order)
    used = s.kernel()
    assert used[0] == getattr(mmf, "KERNEL_" + kind)
    s.set_kernel(used[0])
    assert s.kernel() == used
    s.close()


def test_bricks_are_refused_where_they_do_not_apply(mmf):
    def refused(s):
        with pytest.raises(mmf.MMFError) as e:
            s.set_kernel(mmf.KERNEL_BRICK)
        return e.value.status == mmf.ERR_INVALID

    s = mmf.Solver(2, [100, 90], [0.0] * 3, 0.01, [0] * 4, None, 2)
    assert refused(s)  # its bricks are of the tile kind
    s.close()
    box = [[0.3, 0.2, 0.01, 0.45, 0.4, 0.1]]
    s = mmf.Solver(3, [90, 70, 8], [0.0] * 3, 0.01, [0] * 6, None, 2)
    s.set_kernel(mmf.KERNEL_BRICK)
    s.set_bodies(boxes=box)
    assert s.kernel()[0] == mmf.KERNEL_GATHER
    assert refused(s)
    s.close()
    s = mmf.Solver(3, [90, 70, 8], [0.0] * 3, 0.01, [0] * 6, None, 1)
    s.set_bodies(boxes=box)
    s.set_kernel(mmf.KERNEL_BRICK)
    assert s.kernel()[0] == mmf.KERNEL_BRICK
    solved = (s.cell_flags() & 2 != 0).astype(np.uint8)
    solved[:8] = 0  # ghost cells: fluid, not solved
    s.set_cell_flags((s.cell_flags() & 1).astype(np.uint8), solved)
    assert s.kernel()[0] == mmf.KERNEL_GATHER
    assert refused(s)
    s.close()
