"""The network's gradient kernels where their tiles and sums change: grids of
one row or column (every tap wraps or falls outside), cells just below, at and
past a tile of the weight gradient, batches whose tiles cross samples, and
partial sums that do not divide by the reduction's groups; each layer's
weights and biases against the CPU reference, which rounds to bfloat16 at the
same points, within the float32 accumulation and the activations that fall on
the other side of a rounding (2^-8 relative each, a few percent of them)."""
import numpy as np
import pytest

from tests import surrogate_ref as R
from tests.test_gpu_surrogate import rand_case, to_gpu

pytestmark = pytest.mark.gpu

CASES = [(1, 40, True, False, 1), (40, 1, False, True, 3), (127, 1, True, True, 1), (16, 8, False, False, 1),
         (3, 43, True, False, 1), (11, 23, True, False, 9), (40, 64, True, True, 3)]


@pytest.mark.parametrize("X,Y,perx,pery,B", CASES)
def test_gradient_of_each_layer(X, Y, perx, pery, B):
    from src_incompressible_openmp_amd import surrogate as S

    theta = R.init_params(31)
    f, t = rand_case(X + Y, X, Y, B)
    net = S.Net(X, Y, perx, pery, max_batch=B)
    net.set_params(theta)
    loss, g = net.loss_grad(to_gpu(f), to_gpu(t))
    lref, gref, _ = R.loss_and_grad(theta, f.astype(np.float32), t.astype(np.float32), perx, pery, bf=True)
    assert abs(loss - lref) <= 1e-3 * lref
    o = 0
    for co, _, ci in R.layer_shapes():
        for k in (co * 9 * ci, co):
            assert np.linalg.norm(g[o:o + k] - gref[o:o + k]) <= 3e-2 * np.linalg.norm(gref[o:o + k]), (co, ci, k)
            o += k
    out = net.forward(to_gpu(f))
    net1 = S.Net(X, Y, perx, pery, max_batch=1)
    net1.set_params(theta)
    assert np.array_equal(out, net1.forward(to_gpu(f)))  # one sample at a time: the same bits
