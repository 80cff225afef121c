"""Plans whose spectra or their workspace do not fit: the direct products take
over, with the results, bit by bit, of a plan on which the fast correlation is
switched off.  The failures are forced on the host, before hipMalloc."""
import pytest

from comp_ui_toolbox_amd import BornError, OperatorBatch, OperatorBorn, _lib
from tests.test_fft_gpu import make
from tests.test_kernels_taken_gpu import spec_3d

pytestmark = pytest.mark.gpu

COMMON = 3     # allocations of a workspace that all kernels need


def fail_at(k):
    _lib.lib().born_debug_fail_allocation(k)


def live():
    return _lib.lib().born_debug_live_allocations()


@pytest.fixture(params=["fp32", "split_bf16", "3d"])
def create(request, torch_cuda):
    spec = spec_3d(20, 3, 24, 9, 3, 2, 3, 2) if request.param == "3d" else make(33, 130, 5, 4, 3, 2)
    yield lambda: OperatorBorn.from_sequence(spec, precision="fp32" if request.param == "3d" else request.param)
    fail_at(-1)


def results(op, n_rhs, k=-1):
    """Forward and adjoint of fixed inputs, the k-th allocation of the forward failing."""
    import torch
    gen = torch.Generator(device="cuda:0").manual_seed(n_rhs)
    g = torch.view_as_complex(torch.randn(n_rhs, op.N_points, 2, generator=gen, device="cuda:0"))
    u = torch.view_as_complex(torch.randn(n_rhs, op.N_observations, 2, generator=gen, device="cuda:0"))
    fail_at(k)
    out = op.forward_dev(g)
    fail_at(-1)
    return out, op.adjoint_dev(u)


def same(a, b):
    import torch
    return all(torch.equal(x, y) for x, y in zip(a, b))


def expected(create, n_rhs):
    """Results and live allocations of either kind."""
    out = {}
    for kind in ("direct", "fast"):
        op = create()
        op.set_correlation(kind == "fast")
        before = live()
        out[kind] = results(op, n_rhs), live() - before
        assert op.kernels["pair"] == kind
        op.close()
    assert not same(out["direct"][0], out["fast"][0])
    return out


def test_creation(create):
    """An allocation that fails at creation either is an error that leaves
    nothing behind or one of the spectra, which the first workspace builds."""
    one = expected(create, 1)
    base = live()
    whole = create()
    held = live() - base
    whole.close()
    errors = fallbacks = 0
    for k in range(200):
        fail_at(k)
        try:
            op = create()
        except BornError as e:
            assert e.identifier == "born:OutOfMemory" and live() == base
            errors += 1
            continue
        finally:
            fail_at(-1)
        if live() - base == held:
            break
        fallbacks += 1
        assert same(results(op, 1), one["fast"][0]) and op.kernels["pair"] == "fast"
        op.close()
        assert live() == base
    assert k < 199 and errors >= 10 and fallbacks >= 3
    op.close()


@pytest.mark.parametrize("n_rhs", [1, 3])
def test_first_workspace(create, n_rhs):
    ref, after = expected(create, n_rhs), expected(create, n_rhs + 1)
    base = live()
    for k in range(COMMON, 40):
        op = create()
        op.set_correlation(False)
        op.set_correlation(True)      # the spectra come with the workspace
        before = live()
        assert same(results(op, n_rhs, k), ref[op.kernels["pair"]][0])
        if op.kernels["pair"] == "fast":
            break
        assert live() - before <= ref["direct"][1] + 1      # (the record of a launch that was not to be)
        assert same(results(op, n_rhs), ref["direct"][0])
        assert same(results(op, n_rhs + 1), after["fast"][0])   # the next workspace tries again
        op.close()
        assert live() == base
    assert k > COMMON + 4
    op.close()


def test_later_workspace(create):
    """With the spectra there, a failure of the fast correlation's own buffers
    gives them up; one of the common buffers, with memory to spare, is an error."""
    one, two = expected(create, 1), expected(create, 2)
    base = live()
    for k in range(40):
        op = create()
        assert same(results(op, 1), one["fast"][0])
        if k < COMMON:
            with pytest.raises(BornError, match="born:OutOfMemory"):
                results(op, 2, k)
            fail_at(-1)
        assert same(results(op, 2, -1 if k < COMMON else k), two[op.kernels["pair"]][0])
        if k >= COMMON and op.kernels["pair"] == "fast":
            break
        assert op.kernels["pair"] == ("fast" if k < COMMON else "direct")
        op.close()
        assert live() == base
    assert k > COMMON
    op.close()


def test_batch(create):
    """A batch with a plan that fell back."""
    import torch
    one = expected(create, 1)
    a, b = create(), create()
    results(b, 1, COMMON)
    B = OperatorBatch([a, b])
    assert [a.kernels["pair"], b.kernels["pair"]] == ["fast", "direct"]
    g = torch.ones(a.N_points, dtype=torch.complex64, device="cuda:0")
    us = B.forward_dev([g, g])
    for op, u in zip((a, b), us):
        assert float((u - op.forward_dev(g)).norm() / u.norm()) < 1e-6     # (other work splits)
    assert same(results(a, 1), one["fast"][0]) and same(results(b, 1), one["direct"][0])
    B.close()
