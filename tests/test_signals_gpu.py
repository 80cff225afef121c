"""Time gain compensation and time-domain signals (born_signals.hip) at the
edges of their tiles, against numpy in FP64.

Tolerances: a sum of n FP32 products accumulated in FP32 lies within
(n + 4) 2^-24 of the sum of the products' magnitudes (2^-53 for the FP64
entry); the phase factors of the signals add 3 * 2^-24 per product."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import BornError, OperatorBorn
from comp_ui_toolbox_amd import configs as C
from tests.test_oracle import mixed_tiny_tables

pytestmark = pytest.mark.gpu


def operator(nf, ne=3):
    arr = C.ArraySpec((ne,), (3e-4,), (2.7e-4,), (2,))
    fov = C.FovSpec((9, 2), (7.5e-5, 7.5e-5), 2e-3)
    med = C.MediumSpec()
    waves = [C.qpw_wave(arr, a, med.c_avg) for a in (0.0, 0.1)]
    spec = C.SequenceSpec("s", arr, med, fov, 2e6 + 1e4 * np.arange(nf), waves, [C.identity_mixes(ne) for _ in waves])
    return OperatorBorn.from_sequence(spec)


@pytest.mark.parametrize("nf,M", [(1, 0), (64, 3), (65, 64), (128, 119), (129, 120), (192, 10), (257, 66), (256, 255),
                                  (320, 121), (321, 30), (385, 384), (513, 17)])
def test_tgc_tiles(torch_cuda, nf, M):
    import torch
    op = operator(nf)
    rng = np.random.Generator(np.random.PCG64(nf))
    kernels = [rng.standard_normal(2 * m + 1) + 1j * rng.standard_normal(2 * m + 1) for m in [M] * 5 + [M // 3]]
    op.set_tgc(kernels)
    u = (rng.standard_normal((2, op.N_observations)) + 1j * rng.standard_normal((2, op.N_observations))).astype(np.complex64)
    dev = torch.tensor(u, device="cuda:0")
    i = np.arange(nf)
    for mode in (1, 2):
        y32 = op.tgc_dev(dev, mode=mode).cpu().numpy()
        y64 = (op.tgc_forward if mode == 1 else op.tgc_adjoint)(u.T.astype(np.complex128)).T
        for mk, k in enumerate(kernels):
            m = (len(k) - 1) // 2
            d = i[:, None] - i[None, :]
            A = np.where(np.abs(d) <= m, k[np.clip(d + m, 0, 2 * m)], 0)
            A = A if mode == 1 else A.conj().T
            for r in range(2):
                x = u[r, mk * nf:(mk + 1) * nf].astype(np.complex128)
                ref, size = A @ x, np.abs(A) @ np.abs(x)
                n = 2 * (2 * m + 1) + 4
                assert np.all(np.abs(y32[r, mk * nf:(mk + 1) * nf] - ref) <= n * 2.0 ** -24 * size)
                assert np.all(np.abs(y64[r, mk * nf:(mk + 1) * nf] - ref) <= 2 * n * 2.0 ** -53 * size)


@pytest.mark.parametrize("nf,q0,dq,more", [(1, 3, 1, 1), (2, 0, 5, 1), (9, 0, 1, 1), (17, 5, 3, 1), (33, 7, 1, 3), (64, 1, 2, 1)])
@pytest.mark.parametrize("n_rhs", [1, 3])
def test_time_signals_regular(torch_cuda, nf, q0, dq, more, n_rhs):
    """Zero and Nyquist indices, steps over 1, rows and samples that do not
    fill a wave's block; more: finer sampling than the default."""
    import torch
    op = operator(nf)
    rng = np.random.Generator(np.random.PCG64(nf))
    u = (rng.standard_normal((n_rhs, op.N_observations)) + 1j * rng.standard_normal((n_rhs, op.N_observations))).astype(np.complex64)
    q = q0 + dq * np.arange(nf)
    df = 1e4
    n_t = 2 * q[-1] * more
    rf, got = op.time_signals(torch.tensor(u, device="cuda:0"), df * q, delta_f=df, delta_t=1.0 / (df * n_t))
    assert got == n_t
    x = u.reshape(n_rhs, 6, nf).astype(np.complex128)
    spec = np.zeros((n_rhs, 6, n_t // 2 + 1), dtype=np.complex128)
    spec[..., q] = x
    ref = np.fft.irfft(spec, n=n_t) * n_t
    size = 2.0 * np.abs(x).sum(axis=2, keepdims=True)
    assert np.all(np.abs(rf.cpu().numpy() - ref) <= (2 * nf + 12) * 2.0 ** -24 * size)


@pytest.mark.parametrize("sparse", [0, 5])
@pytest.mark.parametrize("n_rhs", [0, 1, 3])
def test_operator_with_time_gain_in_one_call(torch_cuda, n_rhs, sparse):
    """op_A with time gain gives the values of the two calls bit for bit:
    dense and few occupied points, one vector and matrices, nothing occupied,
    and calls that grow and reuse the staging."""
    _, T = mixed_tiny_tables(distinct=True)
    op = OperatorBorn.from_tables(T)
    with pytest.raises(BornError):
        op.op_A(np.ones(op.N_points), 1, tgc=True)
    rng = np.random.Generator(np.random.PCG64(3))
    op.set_tgc([rng.standard_normal(5) + 1j * rng.standard_normal(5) for _ in op.meta["mix_n_obs"]])
    op.set_sparse_forward(sparse)
    shape = lambda n: (n,) if n_rhs == 0 else (n, n_rhs)
    x = rng.standard_normal(shape(op.N_points)) + 1j * rng.standard_normal(shape(op.N_points))
    few = np.zeros_like(x)
    few[2:4] = x[2:4]
    y = rng.standard_normal(shape(op.N_observations)) + 1j * rng.standard_normal(shape(op.N_observations))
    for g in (few, x, np.zeros_like(x), few):
        u = op.op_A(g, 1, tgc=True)
        assert u.shape == shape(op.N_observations)
        assert np.array_equal(u, op.tgc_forward(op.forward(g)))
        assert np.any(u) == np.any(g)
    back = op.op_A(y, 2, tgc=True)
    assert np.array_equal(back, op.adjoint(op.tgc_adjoint(y)))


@pytest.mark.parametrize("n_t", [21, 126, 127, 128, 129, 130, 257])
def test_time_signals_sample_counts(torch_cuda, n_t):
    """Even and odd numbers of samples around whole wave blocks of sample pairs;
    the bound of test_time_signals_regular."""
    import torch
    nf, q = 10, np.arange(10)
    op = operator(nf)
    rng = np.random.Generator(np.random.PCG64(n_t))
    u = (rng.standard_normal((1, op.N_observations)) + 1j * rng.standard_normal((1, op.N_observations))).astype(np.complex64)
    rf, got = op.time_signals(torch.tensor(u, device="cuda:0"), 1e4 * q, delta_f=1e4, delta_t=1.0 / (1e4 * n_t))
    assert got == n_t
    x = u.reshape(1, 6, nf).astype(np.complex128)
    spec = np.zeros((1, 6, n_t // 2 + 1), dtype=np.complex128)
    spec[..., q] = x
    ref = np.fft.irfft(spec, n=n_t) * n_t
    size = 2.0 * np.abs(x).sum(axis=2, keepdims=True)
    assert np.all(np.abs(rf.cpu().numpy().reshape(ref.shape) - ref) <= (2 * nf + 12) * 2.0 ** -24 * size)
