"""Host arrays to the device and back around the sizes where a copy is cut into
chunks (8 MiB down, 10 MiB up: 524,288 and 655,360 particles of two doubles),
at sizes that leave partial chunks, from one thread and from several with an
object each: every byte."""
import ctypes
import threading

import numpy as np
import pytest

from src_incompressible_openmp_amd.params import poiseuille_params, to_struct
from tests.test_zz_no_alloc import hip_runtime

pytestmark = pytest.mark.gpu


def round_trip(n, seed):
    from src_incompressible_openmp_amd import gpu

    p = to_struct(poiseuille_params(Nx=64, Ny=32, gamma=n / 2048.0))
    p.n = n
    rng = np.random.default_rng(seed)
    x = rng.random((n, 2)) * np.array([p.Lx, p.Ly]) * 0.999
    v = rng.normal(size=(n, 2))
    sim = gpu.Sim(p)
    bad = 0
    for k in range(2):
        v = v + k
        sim.set_state(x, v)
        x2, v2 = sim.get_state()
        bad += not (np.array_equal(x2.reshape(n, 2), x) and np.array_equal(v2.reshape(n, 2), v))
    sim.close()
    return bad


@pytest.mark.parametrize("n", [524287, 524288, 524289, 1048576, 1300001])
def test_round_trip(n):
    assert round_trip(n, n) == 0


def test_several_threads():
    bad = [1] * 4

    def run(k):
        bad[k] = round_trip(600001 + 65536 * k, k)

    th = [threading.Thread(target=run, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert bad == [0] * 4


@pytest.mark.parametrize("up", ["pageable", "pinned"])
@pytest.mark.parametrize("down", ["pageable", "pinned"])
def test_each_direction_alone(up, down):
    """Pinned arrays are copied in one piece and pageable ones in chunks, so
    with one of each only one direction is cut into chunks."""
    from src_incompressible_openmp_amd import gpu

    n = 1200001
    p = to_struct(poiseuille_params(Nx=64, Ny=32, gamma=n / 2048.0))
    p.n = n
    rng = np.random.default_rng(5)
    x = rng.random((n, 2)) * np.array([p.Lx, p.Ly]) * 0.999
    v = rng.normal(size=(n, 2))
    hip = hip_runtime(gpu)
    pinned = []

    def new(kind):
        if kind == "pageable":
            return np.zeros((n, 2))
        q = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(q), ctypes.c_size_t(16 * n), ctypes.c_uint(0)) == 0
        pinned.append(q)
        return np.ctypeslib.as_array(ctypes.cast(q, ctypes.POINTER(ctypes.c_double)), shape=(n, 2))

    hx, hv, x2, v2 = new(up), new(up), new(down), new(down)
    hx[:], hv[:], x2[:], v2[:] = x, v, 0.0, 0.0
    ptr = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    sim = gpu.Sim(p)
    sim.set_state(hx, hv)
    gpu._check(gpu.load().mpcd_gpu_sim_get_state(sim._h, ptr(x2), ptr(v2)))
    sim.close()
    same = np.array_equal(x2, x) and np.array_equal(v2, v)
    for q in pinned:
        assert hip.hipHostFree(q) == 0
    assert same


@pytest.mark.parametrize("grid", [(1024, 1023), (1025, 1024), (2048, 1025)])
def test_large_field_grids(oracle, grid):
    """Field grids of doubles just below and above the size that is cut, and
    one whose counts are cut too, from both entry points that return them."""
    from src_incompressible_openmp_amd import gpu

    nx, ny = grid
    p = to_struct(poiseuille_params(Nx=nx, Ny=ny, gamma=0.25))
    p.n = 200003
    rng = np.random.default_rng(7)
    x = (rng.random((p.n, 2)) * np.array([p.Lx, p.Ly]) * 0.999).reshape(-1)
    v = rng.normal(size=2 * p.n)
    rt = p.gamma / ((p.Lx / p.Nx) * (p.Ly / p.Ny))
    want = oracle.cell_fields(p, x, v, rt)
    sim = gpu.Sim(p)
    sim.set_state(x, v)
    both = gpu.compute_cell_fields(p, x, v, rt), sim.cell_fields(rt)
    sim.close()
    bits = lambda a: np.ascontiguousarray(a).view(np.uint8)
    differ = [k for got in both for k in want if not np.array_equal(bits(got[k]), bits(want[k]))]
    assert not differ
