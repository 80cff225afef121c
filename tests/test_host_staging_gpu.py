"""Host calls of changing size on one plan: the staging kept with it grows with
a call, and is given back after 16 calls that need less than an eighth of it."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBorn
from tests.test_fft_gpu import make

pytestmark = pytest.mark.gpu


def test_sizes(torch_cuda):
    op = OperatorBorn.from_sequence(make(17, 200, 60, 2, 9, 2))
    op.set_sparse_forward(0)
    rng = np.random.Generator(np.random.PCG64(1))
    g = rng.standard_normal((op.N_points, 600)) + 1j * rng.standard_normal((op.N_points, 600))
    few = [op.forward(g[:, :2]), op.adjoint(op.forward(g[:, :2]))]
    many = op.forward(g)                      # 57.6 MB of points
    for k in range(40):                       # 0.2 MB
        u = op.forward(g[:, :2])
        assert np.array_equal(u, few[0]) and np.array_equal(op.adjoint(u), few[1]), k
    assert np.array_equal(op.forward(g), many)
