"""States written through the device view (mmf_get_device_state) between calls:
the next step's dt, the steps and the stage maxima are those of the state that
is there, as after a set_state of it, bit for bit, with every kernel that knows
dt before its first stage."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # name, dim, cells, kernel, body
    ("2d one launch per step", 2, (60, 50), "AUTO", None),
    ("2d bricks", 2, (300, 260), "AUTO", None),
    ("2d bricks, body", 2, (90, 70), "AUTO", {"boxes": [[0.3, 0.2, -1.0, 0.45, 0.4, 1.0]]}),
    ("2d strips", 2, (300, 260), "MARCH", None),
    ("2d gather", 2, (60, 50), "GATHER", None),
    ("3d bricks", 3, (20, 18, 12), "AUTO", None),
    ("3d marching", 3, (64, 16, 16), "MARCH", None),
    ("3d marching, reflecting", 3, (64, 17, 11), "MARCH", None),
    ("3d marching, body", 3, (64, 16, 16), "MARCH", {"boxes": [[0.3, 0.05, 0.05, 0.45, 0.1, 0.1]]}),
]


class Planes:
    """The SoA planes at a device address; writes rows [cells][5]."""

    def __init__(self, address, stride):
        self.L = C.CDLL("libamdhip64.so.7")
        self.L.hipMemcpy.argtypes = [C.c_void_p, C.c_void_p, C.c_size_t, C.c_int]
        self.address, self.stride = address, stride

    def write(self, U):
        for k in range(5):
            a = np.ascontiguousarray(U[:, k])
            assert self.L.hipMemcpy(self.address + 8 * k * self.stride, a.ctypes.data, a.nbytes, 1) == 0
        assert self.L.hipDeviceSynchronize() == 0


def flow(N, seed, p):
    r = np.random.default_rng(seed)
    U = np.zeros((N, 5))
    U[:, 0] = r.uniform(0.9, 1.1, N)
    U[:, 1:3] = r.uniform(-0.1, 0.1, (N, 2))
    U[:, 4] = p * r.uniform(0.9, 1.1, N) / 0.4 + 0.05
    return U


def solver(mmf, name, dim, n, kernel, body):
    bc = [1] * 6 if "reflecting" in name else [0] * 6
    s = mmf.Solver(dim, list(n), [0.0] * 3, 0.5 / max(n), bc, None, 1)
    s.set_kernel(getattr(mmf, "KERNEL_" + kernel))
    if body:
        s.set_bodies(**body)
    return s


@pytest.mark.parametrize("name,dim,n,kernel,body", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("loop", ["advance", "run"])
def test_state_written_through_the_view(mmf, name, dim, n, kernel, body, loop):
    N = int(np.prod(n))
    states = [flow(N, 1, 1.0), flow(N, 2, 9.0), flow(N, 3, 0.3), flow(N, 4, 4.0)]
    out = []
    for through_view in (True, False):
        s = solver(mmf, name, dim, n, kernel, body)
        s.set_state(states[0])
        s.set_time(0.0, 1e30, 0.3)
        # one address, taken before any step
        planes = Planes(*s.device_state(mmf.STATE_U)) if through_view else None
        seen = []
        # a graph's worth of steps, then few
        for k, steps in enumerate((20, 3, 2, 1)):
            if k:
                s.synchronize()
                if through_view:
                    planes.write(states[k])
                else:
                    s.set_state(states[k])
            if loop == "run":
                s.run(max_steps=steps)
            else:
                s.advance(steps)
            t, dt, step, eig = s.time()
            seen.append((t, dt, step, tuple(eig), s.get_state().tobytes()))
        out.append(seen)
        s.close()
    for k, (a, b) in enumerate(zip(*out)):
        assert a[:4] == b[:4], (name, k, a[:4], b[:4])
        assert a[4] == b[4], (name, k)
