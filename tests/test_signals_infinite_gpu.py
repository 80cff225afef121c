"""Time signals of spectra with infinite coefficients at the indices that count
once: their samples are infinite, of the coefficient's sign, not undefined."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBorn
from tests.test_fft_gpu import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q0,at", [(0, 0), (2, 7)])
def test_infinite_coefficient(torch_cuda, q0, at):
    torch = torch_cuda
    spec = make(5, 20, 2, 2, 8, 1)
    spec.frequencies = 1e6 * (q0 + np.arange(8))
    if q0 == 0:       # (a medium has no zero frequency: the axis is the caller's)
        spec.frequencies = 1e6 * (1 + np.arange(8))
    op = OperatorBorn.from_sequence(spec)
    axis = 1e6 * (q0 + np.arange(8))
    u = torch.view_as_complex(torch.randn(op.N_observations // 8, 8, 2, device="cuda:0"))
    u[::2, at] = torch.inf
    rf, n_t = op.time_signals(u.reshape(-1), axis, delta_f=1e6)
    assert n_t == 2 * (q0 + 7)
    assert torch.isfinite(rf[0, 1::2]).all()
    sign = torch.tensor([1.0 if at == 0 or n % 2 == 0 else -1.0 for n in range(n_t)], device="cuda:0")
    assert torch.equal(rf[0, ::2], (sign * torch.inf).expand_as(rf[0, ::2]))
