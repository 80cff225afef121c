"""Fast lateral correlation of 2-D plans (born_fft.hip) against the FP64
oracle and the general gather path, at the sizes where its transforms,
segments and slots have edges: transform lengths 64, 128 and 256 and the
element counts beside them, one and several segments per row, rows whose
points per phase differ, points per pitch that do not divide a wave's slots,
slot counts that leave padding, one column, several right-hand sides.

Tolerance: three FP32 transforms of at most 256 points (the spectra's
rounding, the data, the way back) of at most 8 stages each give a relative L2
error below 3 * 8 * 2^-24 = 1.5e-6 in the worst case and about its square
root of 24 part of it, 3e-7, for independent roundings; 1e-6 is taken."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBorn
from comp_ui_toolbox_amd import configs as C
from oracle import born_oracle as O
from tests.test_oracle import mixed_tiny_tables

pytestmark = pytest.mark.gpu

TOL = 1e-6


def make(ne, nx, nz, npp, nf, waves, n_mix=0):
    pitch = 3e-4
    arr = C.ArraySpec((ne,), (pitch,), (2.7e-4,), (2,))
    med = C.MediumSpec()
    fov = C.FovSpec((nx, nz), (pitch / npp, pitch / npp), 2e-3)
    rng = np.random.Generator(np.random.PCG64(ne * 1000 + nx))
    ws = [C.random_wave(arr, rng, 1e-6) for _ in range(waves)]
    mixes = [[C.MixSpec(np.arange(ne), np.where(rng.random(ne) < 0.5, -1.0, 1.0)) for _ in range(n_mix)]
             if n_mix else C.identity_mixes(ne) for _ in ws]
    return C.SequenceSpec("fft", arr, med, fov, np.linspace(2e6, 6e6, nf), ws, mixes)


# elements, points x, z, points per pitch, frequencies, waves, mixes, rhs
SIZES = [
    (1, 5, 3, 1, 2, 1, 0, 1),          # one element, padding slots, one wave
    (2, 9, 1, 4, 1, 1, 0, 2),          # one row
    (17, 70, 5, 2, 3, 2, 0, 1),        # length 64
    (48, 130, 7, 2, 2, 3, 0, 3),       # several segments or a longer transform
    (64, 257, 3, 4, 3, 2, 0, 1),       # 65 points in phase 0, 64 in the others
    (65, 250, 5, 4, 2, 3, 3, 2),       # one element over half of 128
    (100, 301, 4, 2, 3, 7, 0, 1),      # more than half full
    (127, 516, 2, 4, 2, 2, 0, 1),      # 129 points per phase: the length 256 exactly full
    (128, 512, 2, 4, 2, 17, 0, 1),     # 128 points per phase
    (128, 700, 3, 4, 2, 1, 0, 1),      # two segments of unequal use
    (33, 101, 6, 3, 3, 2, 0, 2),       # phases that do not divide the slots of a wave
    (20, 77, 3, 5, 2, 2, 2, 1),
    (31, 40, 9, 1, 3, 2, 0, 1),        # field of view narrower than the aperture, one point per pitch
    # the remaining counts of entries per lane (4 to 16) of each length
    (27, 30, 3, 1, 2, 2, 0, 1), (13, 134, 3, 1, 2, 2, 0, 2), (6, 214, 2, 2, 2, 2, 0, 1),       # 64: 8, 12, 16
    (91, 36, 3, 3, 2, 2, 0, 1), (70, 90, 3, 1, 2, 2, 0, 2), (32, 176, 2, 1, 2, 2, 0, 1),       # 128: 4, 6, 12
    (17, 402, 2, 2, 2, 2, 0, 1),                                                              # 128: 16
    (98, 63, 3, 1, 2, 2, 0, 2), (61, 353, 2, 2, 2, 2, 0, 1), (33, 209, 3, 1, 2, 2, 0, 1),      # 256: 4, 12, 16
]


@pytest.mark.parametrize("ne,nx,nz,npp,nf,waves,n_mix,n_rhs", SIZES)
def test_against_oracle_and_general_path(torch_cuda, ne, nx, nz, npp, nf, waves, n_mix, n_rhs):
    import torch
    spec = make(ne, nx, nz, npp, nf, waves, n_mix)
    T = O.direct_tables(spec)
    op = OperatorBorn.from_sequence(spec)
    assert op.path == "structured"
    rng = np.random.Generator(np.random.PCG64(7))
    g = rng.standard_normal((n_rhs, op.N_points)) + 1j * rng.standard_normal((n_rhs, op.N_points))
    u = rng.standard_normal((n_rhs, op.N_observations)) + 1j * rng.standard_normal((n_rhs, op.N_observations))
    gd = torch.tensor(g.astype(np.complex64), device="cuda:0")
    ud = torch.tensor(u.astype(np.complex64), device="cuda:0")
    fast = [op.forward_dev(gd).cpu().numpy(), op.adjoint_dev(ud).cpu().numpy()]
    again = [op.forward_dev(gd).cpu().numpy(), op.adjoint_dev(ud).cpu().numpy()]
    op.force_general(True)
    general = [op.forward_dev(gd).cpu().numpy(), op.adjoint_dev(ud).cpu().numpy()]
    for r in range(n_rhs):
        ref = [O.forward(T, gd[r].cpu().numpy()), O.adjoint(T, ud[r].cpu().numpy())]
        for k in range(2):
            assert np.array_equal(fast[k][r], again[k][r])
            assert O.rel_l2(fast[k][r], ref[k].reshape(-1)) < TOL, ("oracle", k)
            assert O.rel_l2(fast[k][r], general[k][r]) < 2 * TOL, ("general", k)


def test_lists_of_unequal_length(torch_cuda):
    """Un-mixing lists of 0 to 11 entries side by side, 5 on average."""
    spec = make(20, 60, 3, 2, 3, 2, 5)
    rng = np.random.Generator(np.random.PCG64(4))
    for k, mixes in enumerate(spec.mixes):
        for n in (3, 7, 12, 20, 20, 20):
            e = rng.permutation(np.arange(1, 20))[:min(n, 19)]   # element 0 in the dense mixes only
            mixes.append(C.MixSpec(e, rng.standard_normal(len(e)), np.array([k, 2])))
    T = O.direct_tables(spec)
    op = OperatorBorn.from_sequence(spec)
    u = rng.standard_normal(op.N_observations) + 1j * rng.standard_normal(op.N_observations)
    assert O.rel_l2(op.adjoint(u), O.adjoint(T, u).reshape(-1)) < TOL


def test_mixed_tables_and_zero_columns(torch_cuda):
    """Frequency subsets, repeated frequencies and a right-hand side that is
    zero, from an operator's own tables."""
    _, T = mixed_tiny_tables()
    op = OperatorBorn.from_tables(T)
    rng = np.random.Generator(np.random.PCG64(8))
    g = rng.standard_normal((op.N_points, 3)) + 1j * rng.standard_normal((op.N_points, 3))
    g[:, 1] = 0
    u = op.forward(g)
    for r in range(3):
        ref = O.forward(T, g[:, r]).reshape(-1)
        assert np.all(u[:, r] == 0) if r == 1 else O.rel_l2(u[:, r], ref) < TOL


# elements x, y, points x, y, z, points per pitch, frequencies, waves, rhs
SIZES_3D = [
    (4, 3, 19, 7, 3, 2, 2, 2, 1),      # 64 x 64, both phases of x in one tile
    (32, 2, 66, 9, 2, 2, 2, 1, 2),     # 33 points per phase: more than half full
    (20, 8, 70, 25, 5, 2, 1, 2, 1),
    (32, 4, 72, 20, 2, 2, 1, 2, 3),    # 128 x 64
    (3, 33, 10, 68, 2, 2, 2, 1, 1),    # 64 x 128
    (34, 33, 64, 66, 1, 2, 1, 2, 1),   # 128 x 128, just over 64 on both axes
    (5, 4, 40, 30, 9, 1, 2, 1, 2),     # one point per pitch
    (6, 5, 50, 31, 2, 3, 2, 2, 1),     # three phases
    (17, 2, 101, 5, 2, 4, 1, 1, 1),    # four phases, field of view wider than the aperture
]


@pytest.mark.parametrize("nex,ney,nx,ny,nz,npp,nf,waves,n_rhs", SIZES_3D)
def test_volume(torch_cuda, nex, ney, nx, ny, nz, npp, nf, waves, n_rhs):
    """Planes: two more transforms of at most 7 stages, worst case
    3 * 14 * 2^-24 = 2.5e-6; 1.5e-6 is taken."""
    import torch
    pitch = 3e-4
    arr = C.ArraySpec((nex, ney), (pitch, pitch), (2.7e-4, 2.7e-4), (2, 2))
    fov = C.FovSpec((nx, ny, nz), (pitch / npp,) * 3, 3e-3)
    rng = np.random.Generator(np.random.PCG64(nex * 100 + ny))
    ws = [C.random_wave(arr, rng, 1e-6) for _ in range(waves)]
    spec = C.SequenceSpec("fft3", arr, C.MediumSpec(), fov, np.linspace(2.5e6, 4e6, nf), ws,
                          [C.identity_mixes(nex * ney) for _ in ws])
    T = O.direct_tables(spec)
    op = OperatorBorn.from_sequence(spec)
    assert op.path == "structured"
    g = rng.standard_normal((n_rhs, op.N_points)) + 1j * rng.standard_normal((n_rhs, op.N_points))
    u = rng.standard_normal((n_rhs, op.N_observations)) + 1j * rng.standard_normal((n_rhs, op.N_observations))
    gd = torch.tensor(g.astype(np.complex64), device="cuda:0")
    ud = torch.tensor(u.astype(np.complex64), device="cuda:0")
    fast = [op.forward_dev(gd).cpu().numpy(), op.adjoint_dev(ud).cpu().numpy()]
    assert np.array_equal(fast[0], op.forward_dev(gd).cpu().numpy())
    assert np.array_equal(fast[1], op.adjoint_dev(ud).cpu().numpy())
    op.force_general(True)
    general = [op.forward_dev(gd).cpu().numpy(), op.adjoint_dev(ud).cpu().numpy()]
    for r in range(n_rhs):
        ref = [O.forward(T, gd[r].cpu().numpy()), O.adjoint(T, ud[r].cpu().numpy())]
        for k in range(2):
            assert O.rel_l2(fast[k][r], ref[k].reshape(-1)) < 1.5e-6, ("oracle", k)
            assert O.rel_l2(fast[k][r], general[k][r]) < 3e-6, ("general", k)


@pytest.mark.parametrize("ne,nx,nz,npp,nf,waves,n_mix,n_rhs", [
    (8, 16, 400, 2, 2, 1, 0, 1),       # 24 slot blocks of a few values: eight threads per value
    (9, 15, 200, 4, 3, 2, 5, 3),       # the same, several mixes and right-hand sides
    (24, 40, 34, 1, 17, 3, 3, 1),      # columns in several groups per slot group
    (33, 60, 3, 2, 2, 2, 4, 2), (70, 40, 2, 1, 3, 1, 5, 1), (128, 60, 2, 1, 2, 1, 11, 2),      # lists of 4, 5 and 11
])
def test_split_of_small_plans(torch_cuda, ne, nx, nz, npp, nf, waves, n_mix, n_rhs):
    test_against_oracle_and_general_path(torch_cuda, ne, nx, nz, npp, nf, waves, n_mix, n_rhs)


@pytest.mark.parametrize("three", [False, True])
@pytest.mark.parametrize("entry", [1e7, np.inf])
def test_uneven_tables_keep_the_direct_products(torch_cuda, three, entry):
    """One entry of h_ref far above the others (a grid point next to an
    element): what the other entries give has to keep its accuracy, which a
    transform over the row would lose to the rounding of the large one."""
    spec = make(33, 101, 6, 3, 3, 2)
    if three:
        arr = C.ArraySpec((4, 3), (3e-4, 3e-4), (2.7e-4, 2.7e-4), (2, 2))
        waves = [C.random_wave(arr, np.random.Generator(np.random.PCG64(w)), 1e-6) for w in range(2)]
        spec = C.SequenceSpec("fft3", arr, C.MediumSpec(), C.FovSpec((19, 7, 3), (1.5e-4,) * 3, 3e-3),
                              np.linspace(2.5e6, 4e6, 2), waves, [C.identity_mixes(12) for _ in waves])
    T = O.build_tables(spec)
    at = T.N_points // 3
    touched = np.any(np.asarray(T.shift).reshape(T.N_points, -1) - 1 == at, axis=1)
    assert touched.any() and not touched.all()
    clean = T.h_ref.copy()
    T.h_ref[1, at] = entry
    op = OperatorBorn.from_tables(T)
    assert op.path == "structured"
    rng = np.random.Generator(np.random.PCG64(9))
    u = rng.standard_normal(op.N_observations) + 1j * rng.standard_normal(op.N_observations)
    g = rng.standard_normal(op.N_points) + 1j * rng.standard_normal(op.N_points)
    g[touched] = 0
    op.force_general(True)
    general = op.adjoint(u)
    op.force_general(False)
    back = op.adjoint(u)
    T.h_ref = clean
    ref = O.adjoint(T, u).reshape(-1)
    assert O.rel_l2(general[~touched], ref[~touched]) < TOL
    if np.isfinite(entry):
        assert O.rel_l2(back[~touched], ref[~touched]) < TOL
        assert O.rel_l2(op.forward(g), O.forward(T, g).reshape(-1)) < TOL
    else:   # the points whose rows of the table hold no such entry
        plane = T.N_points // spec.fov.N_points_axis[-1]
        rest = np.arange(T.N_points) // plane != at // plane
        assert O.rel_l2(back[rest], ref[rest]) < TOL
