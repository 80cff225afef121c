"""Received energies of rows enough for workgroups of four waves, beside those
of eight, against the map-driven kernel (2e-12, as at fewer rows)."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBorn
from tests.test_fft_gpu import make

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ne,nx,nz,npp", [(65, 384, 256, 4), (65, 384, 257, 4), (24, 250, 300, 4), (24, 250, 520, 4), (20, 500, 270, 2)])
def test_rows(torch_cuda, ne, nx, nz, npp):
    op = OperatorBorn.from_sequence(make(ne, nx, nz, npp, 5, 1))
    assert op.kernels["energy"] == "fast"
    fast = op.energy_rx(0)
    op.force_general(True)
    general = op.energy_rx(0)
    assert np.max(np.abs(fast - general) / general) < 2e-12
