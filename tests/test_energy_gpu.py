"""Received energies of structured plans (born_energy.hip) against the FP64
oracle and the map-driven kernel of the general path, over the sizes where
the fast kernels' lanes, windows and observation groups have edges.

Tolerances: both kernels take FP64 sums of at most 1e4 positive terms of the
same FP32 tables, 1e4 * 2^-53 = 1.1e-12 apart; the tables' rounding to FP32
(2^-24 each in h_ref and p_inc, squared) moves E by at most 4 * 2^-24 = 2.4e-7."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBorn
from comp_ui_toolbox_amd import configs as C
from oracle import born_oracle as O

pytestmark = pytest.mark.gpu


def mixes_of(kind, ne, nf, rng):
    if kind == "single":
        return [C.MixSpec(np.array([e]), np.array([1.0 + 0.1 * e])) for e in range(0, ne, 2)]
    if kind == "dense":
        return [C.MixSpec(np.arange(ne), rng.standard_normal(ne)) for _ in range(5)]
    # both: one element, a sub-aperture on two frequencies, all elements reversed
    return [C.MixSpec(np.array([ne - 1]), np.array([2.0])),
            C.MixSpec(np.arange(ne // 3, ne // 3 + 2) % ne, np.array([1.0, -1.0]), np.array([nf - 1, 0])),
            C.MixSpec(np.arange(ne)[::-1].copy(), rng.standard_normal(ne))]


def check(op, T, measurements, kind):
    for m in range(measurements):
        fast = op.energy_rx(m)
        op.force_general(True)
        general = op.energy_rx(m)
        op.force_general(False)
        ref = O.energy_rx(T, m)
        assert np.max(np.abs(fast - general) / general) < 2e-12
        assert np.linalg.norm(fast - ref) < 2.4e-7 * np.linalg.norm(ref)
        if kind == "single":
            assert np.max(np.abs(fast - ref) / ref) < 2.4e-7


# elements, points x, z, points per pitch
SIZES = [(3, 9, 2, 1), (17, 130, 3, 2), (64, 384, 2, 4), (65, 257, 2, 4), (128, 515, 2, 4), (24, 101, 2, 3), (8, 150, 2, 16),
         # the remaining counts of points and window entries per lane, and a window filled in between
         (20, 512, 2, 4), (128, 512, 2, 4), (9, 380, 2, 4), (128, 240, 2, 5), (64, 150, 2, 16)]


@pytest.mark.parametrize("kind", ["single", "dense", "both"])
@pytest.mark.parametrize("ne,nx,nz,npp", SIZES)
def test_linear_array(torch_cuda, ne, nx, nz, npp, kind):
    pitch, nf = 3e-4, 5
    rng = np.random.Generator(np.random.PCG64(nx))
    arr = C.ArraySpec((ne,), (pitch,), (2.7e-4,), (2,))
    fov = C.FovSpec((nx, nz), (pitch / npp, pitch / npp), 2e-3)
    waves = [C.random_wave(arr, rng, 1e-6) for _ in range(2)]
    spec = C.SequenceSpec("e", arr, C.MediumSpec(), fov, np.linspace(2e6, 5e6, nf), waves,
                          [mixes_of(kind, ne, nf, rng) for _ in waves])
    op = OperatorBorn.from_sequence(spec)
    assert op.path == "structured"
    check(op, O.direct_tables(spec), 2, kind)


@pytest.mark.parametrize("kind", ["single", "both"])
def test_matrix_array(torch_cuda, kind):
    rng = np.random.Generator(np.random.PCG64(5))
    arr = C.ArraySpec((5, 3), (3e-4, 3e-4), (2.7e-4, 2.7e-4), (2, 2))
    fov = C.FovSpec((19, 7, 3), (1.5e-4, 1.5e-4, 1.5e-4), 2e-3)
    waves = [C.qsw_wave(arr, np.array([0.0, 0.0, -5e-3]), 1500.0)]
    spec = C.SequenceSpec("e3", arr, C.MediumSpec(), fov, np.linspace(2e6, 4e6, 3), waves,
                          [mixes_of(kind, 15, 3, rng)])
    op = OperatorBorn.from_sequence(spec)
    assert op.path == "structured"
    check(op, O.direct_tables(spec), 1, kind)


@pytest.mark.parametrize("kind", ["single", "dense"])
@pytest.mark.parametrize("nf,M", [(5, 0), (17, 3), (32, 31), (33, 32), (33, 40), (50, 14), (65, 64), (72, 56), (73, 100),
                                  (128, 127), (129, 128), (129, 100), (200, 56)])
def test_under_tgc(torch_cuda, nf, M, kind):
    """Transform lengths 64, 128 and 256 for the convolution along the
    frequencies, and the odd lengths whose longest lag is taken separately
    (33, 65, 129).  Two FP32 transforms of at most 8 stages, 2 * 8 * 2^-24 =
    9.5e-7 in the compensated rows, twice that in their squares, and the
    tables' 2.4e-7: 2.2e-6."""
    ne, npp = 6, 4
    rng = np.random.Generator(np.random.PCG64(nf + M))
    arr = C.ArraySpec((ne,), (3e-4,), (2.7e-4,), (2,))
    fov = C.FovSpec((37, 3), (3e-4 / npp, 3e-4 / npp), 2e-3)
    waves = [C.random_wave(arr, rng, 1e-6) for _ in range(2)]
    spec = C.SequenceSpec("et", arr, C.MediumSpec(), fov, 2e6 + 3e4 * np.arange(nf), waves,
                          [mixes_of(kind, ne, nf, rng) for _ in waves])
    op = OperatorBorn.from_sequence(spec)
    T = O.direct_tables(spec)
    n_mix = len(spec.mixes[0])
    kernels = [rng.standard_normal(2 * m + 1) + 1j * rng.standard_normal(2 * m + 1)
               for m in ([M] * (2 * n_mix - 1) + [M // 2])]
    op.set_tgc(kernels)
    for m in range(2):
        ref = O.energy_rx(T, m, kernels[m * n_mix:(m + 1) * n_mix])
        E = op.energy_rx(m, tgc=True)
        assert np.linalg.norm(E - ref) < 2.2e-6 * np.linalg.norm(ref)
        assert np.array_equal(E, op.energy_rx_dev(m, tgc=True).cpu().numpy())


@pytest.mark.parametrize("kind", ["single", "dense"])
def test_entry_that_is_not_finite(torch_cuda, kind):
    """A table entry that is not finite stays with the points that see it."""
    rng = np.random.Generator(np.random.PCG64(2))
    arr = C.ArraySpec((17,), (3e-4,), (2.7e-4,), (2,))
    waves = [C.random_wave(arr, rng, 1e-6)]
    spec = C.SequenceSpec("e", arr, C.MediumSpec(), C.FovSpec((130, 3), (1.5e-4, 1.5e-4), 2e-3), np.linspace(2e6, 5e6, 3),
                          waves, [mixes_of(kind, 17, 3, rng)])
    T = O.build_tables(spec)
    at = T.N_points // 3 + 20
    seen = np.any(np.asarray(T.shift) - 1 == at, axis=1)
    ref = O.energy_rx(T, 0)
    T.h_ref[1, at] = np.inf
    op = OperatorBorn.from_tables(T)
    assert op.path == "structured" and seen.any() and not seen.all()
    assert np.linalg.norm((op.energy_rx(0) - ref)[~seen]) < 2.4e-7 * np.linalg.norm(ref[~seen])
