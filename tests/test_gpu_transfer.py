"""Host arrays to the device and back around the size where a copy is cut into
chunks (8 MiB: 524,288 particles of two doubles), at sizes that leave partial
chunks, from one thread and from several with an object each: every byte."""
import threading

import numpy as np
import pytest

from src_incompressible_openmp_amd.params import poiseuille_params, to_struct

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
