"""Energies under time gain where the transforms' roundings do not average out:
sums of squares over thousands of rows keep what is systematic.

FP32 constants and spectra rounded to the nearest lower the energy of the two
transforms by about 1.1e-7 (cos(pi / 8) and sqrt(1 / 2) are both rounded down,
3e-8 per transform, the twiddles' mean magnitude another 1e-8 each, the
spectra's rounding 3e-8), and each of them alone is above the error of the
map-driven kernel, about 2e-8 from the rounding of the taps.  With the
remainders that the kernel carries, 5e-9 per transform are left: it has to be
as close to 64 bits as the map-driven kernel."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBorn
from comp_ui_toolbox_amd import configs as C
from comp_ui_toolbox_amd.tgc import exponential_kernels
from oracle import born_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nf", [65, 100])
def test_sums_of_squares(torch_cuda, nf):
    ne, df = 64, 31.25e3
    arr = C.ArraySpec((ne,), (3.048e-4,), (2.7e-4,), (4,))
    fov = C.FovSpec((96, 12), (7.62e-5,) * 2, 8e-3)
    spec = C.SequenceSpec("a", arr, C.MediumSpec(), fov, 2e6 + df * np.arange(nf), [C.qpw_wave(arr, 0.05, 1500.0)],
                          [C.identity_mixes(ne)])
    op = OperatorBorn.from_sequence(spec)
    kernels = exponential_kernels(1.2e5, np.tile((0.0, 0.9 / df), (ne, 1)), df, -40.0)
    op.set_tgc(kernels)
    assert op.kernels["energy_tgc"] == "fast"
    ref = O.energy_rx(O.direct_tables(spec), 0, kernels)
    e = np.linalg.norm(op.energy_rx(0, tgc=True) - ref) / np.linalg.norm(ref)
    op.force_general(True)
    g = np.linalg.norm(op.energy_rx(0, tgc=True) - ref) / np.linalg.norm(ref)
    print(f"{nf} frequencies: {e:.2e} (map-driven kernel {g:.2e})", flush=True)
    assert e <= g
