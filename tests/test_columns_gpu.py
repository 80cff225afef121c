"""Columns of A on regular structured plans (born_columns.hip) against the
map-driven kernel of the general path, over element blocks, measurement
groups, frequency blocks and point groups with remainders.

Tolerance: both take FP64 sums of the same FP32 tables, at most 40 terms:
40 * 2^-53 = 4.4e-15 of the largest term apart, so 1e-13 of the column's
norm; the device variant rounds to FP32, 2^-24 per component: 2e-7."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBorn
from comp_ui_toolbox_amd import configs as C

pytestmark = pytest.mark.gpu


def build(ne, nx, nz, npp, nf, waves, kind):
    pitch = 3e-4
    rng = np.random.Generator(np.random.PCG64(ne + nx))
    arr = C.ArraySpec((ne,), (pitch,), (2.7e-4,), (2,))
    fov = C.FovSpec((nx, nz), (pitch / npp, pitch / npp), 2e-3)
    ws = [C.random_wave(arr, rng, 1e-6) for _ in range(waves)]
    some = [C.MixSpec(np.arange(ne), rng.standard_normal(ne)) for _ in range(3)]
    sub = [C.MixSpec(np.array([ne - 1, 0]), np.array([1.0, -2.0]))]
    one = [C.MixSpec(np.array([e]), np.array([1.0 + 0.5 * e])) for e in range(ne - 1, -1, -1)]
    mixes = {"single": one, "multi": some + sub, "both": some + one + sub}[kind]
    return C.SequenceSpec("c", arr, C.MediumSpec(), fov, np.linspace(2e6, 5e6, nf), ws, [mixes for _ in ws])


@pytest.mark.parametrize("kind", ["single", "multi", "both"])
@pytest.mark.parametrize("ne,nx,nz,npp,nf,waves", [
    (3, 9, 2, 1, 1, 1), (16, 70, 3, 2, 17, 9), (33, 150, 4, 4, 16, 8), (40, 61, 5, 3, 35, 2)])
@pytest.mark.parametrize("n", [1, 6])
def test_against_general_path(torch_cuda, ne, nx, nz, npp, nf, waves, kind, n):
    op = OperatorBorn.from_sequence(build(ne, nx, nz, npp, nf, waves, kind))
    rng = np.random.Generator(np.random.PCG64(n))
    pts = rng.integers(0, op.N_points, n)
    pts[-1] = op.N_points - 1
    fast, dev = op.columns(pts), op.columns_dev(pts).cpu().numpy().T
    op.force_general(True)
    ref = op.columns(pts)
    for j in range(n):
        norm = np.linalg.norm(ref[:, j])
        assert norm > 0
        assert np.linalg.norm(fast[:, j] - ref[:, j]) < 1e-13 * norm
        assert np.linalg.norm(dev[:, j] - ref[:, j]) < 2e-7 * norm
