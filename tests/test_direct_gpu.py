"""The direct products of structured plans, which serve plans off the fast
correlation: the tests of the few-column, stacked, matrix and split kernels,
of many right-hand sides, of batches and of the autotuner, on plans with the
fast correlation switched off."""
import numpy as np
import pytest

from comp_ui_toolbox_amd import OperatorBatch, OperatorBorn
from comp_ui_toolbox_amd import configs as C
from tests.test_batch_gpu import (fp32_set, inputs, rel, test_batch_against_oracle, test_batch_autotune_keeps_results,  # noqa: F401
                                  test_batch_follows_plan_workspace_changes, test_batch_graph_replay,
                                  test_batch_matches_single_plans, test_batch_split, test_plan_autotune_keeps_results,
                                  uneven_specs)
from tests.test_fft_gpu import make
from tests.test_parity_gpu import (test_3d_geometry_structured, test_few_column_kernels, test_many_rhs,  # noqa: F401
                                   test_many_rhs_many_waves, test_narrow_fov_split_bf16, test_split_small_tables,
                                   test_stacked_mfma_kernels, test_tiny_odd_geometries, test_zero_and_subnormal_input)

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def direct(torch_cuda):
    wrap = OperatorBorn._wrap.__func__

    def without_correlation(cls, *a, **k):
        op = wrap(cls, *a, **k)
        op.set_correlation(False)
        assert op.kernels["pair"] == {"structured": "direct", "general": "gather"}[op.path]
        return op

    with pytest.MonkeyPatch.context() as mp:
        mp.setattr(OperatorBorn, "_wrap", classmethod(without_correlation))
        yield


@pytest.mark.parametrize("graph", [False, True])
def test_batch_of_both_kinds(torch_cuda, graph):
    """Plans on the direct products beside plans on the fast correlation, 2-D
    and 3-D, in one batch: every result is that of the plan alone (other work
    splits, FP32: 1e-6)."""
    torch = torch_cuda
    ops = [OperatorBorn.from_sequence(s) for s in uneven_specs(16)]
    arr = C.ArraySpec((4, 3), (3e-4, 3e-4), (2.7e-4, 2.7e-4), (2, 2))
    waves = [C.random_wave(arr, np.random.Generator(np.random.PCG64(w)), 1e-6) for w in range(2)]
    for n in ((19, 7, 3), (30, 12, 2)):
        ops.append(OperatorBorn.from_sequence(C.SequenceSpec("b3", arr, C.MediumSpec(), C.FovSpec(n, (7.5e-5,) * 3, 3e-3),
                                                             np.linspace(2.5e6, 4e6, 2), waves,
                                                             [C.identity_mixes(12) for _ in waves])))
    ops.append(OperatorBorn.from_sequence(make(15, 60, 3, 4, 3, 2, 5)))
    for op in ops[::2] + [ops[5]]:
        op.set_correlation(True)
    B = OperatorBatch(ops, graph=graph)
    kinds = [op.kernels["pair"] for op in ops]
    assert kinds == ["fast", "direct", "fast", "direct", "fast", "fast", "fast", "direct"]
    g, u = inputs(torch, ops, 31)
    outs = [torch.empty_like(x) for x in u], [torch.empty_like(x) for x in g]
    for rep in range(3):
        for x in outs[0] + outs[1]:
            x.zero_()
        B.forward_dev(g, outs=outs[0])
        B.adjoint_dev(u, outs=outs[1])
        for i, op in enumerate(ops):
            assert rel(outs[0][i], op.forward_dev(g[i])) < 1e-6, (rep, i)
            assert rel(outs[1][i], op.adjoint_dev(u[i])) < 1e-6, (rep, i)
    B.autotune()
    ops[0].set_correlation(False)    # the batch follows
    ops[1].set_correlation(True)
    for x, y in zip(B.forward_dev(g), [op.forward_dev(v) for op, v in zip(ops, g)]):
        assert rel(x, y) < 1e-6
    B.close()


@pytest.mark.parametrize("ne,nx,nz,npp,nf,waves,n_mix,n_rhs", [
    (17, 70, 5, 2, 3, 2, 0, 1), (65, 250, 5, 4, 2, 3, 3, 2), (128, 512, 2, 4, 2, 17, 0, 1), (31, 40, 9, 1, 3, 2, 0, 1)])
def test_both_kinds_agree(torch_cuda, ne, nx, nz, npp, nf, waves, n_mix, n_rhs):
    """Each of the two within its FP32 rounding (1e-6 and 5e-7) of the other,
    and back and forth on one plan."""
    import torch
    op = OperatorBorn.from_sequence(make(ne, nx, nz, npp, nf, waves, n_mix))
    g = torch.view_as_complex(torch.randn(n_rhs, op.N_points, 2, device="cuda:0"))
    u = torch.view_as_complex(torch.randn(n_rhs, op.N_observations, 2, device="cuda:0"))
    out = []
    for on in (False, True, False):
        op.set_correlation(on)
        out.append((op.forward_dev(g), op.adjoint_dev(u)))
        assert op.kernels["pair"] == ("fast" if on else "direct")
    for k in range(2):
        assert torch.equal(out[0][k], out[2][k])
        assert not torch.equal(out[0][k], out[1][k])
        assert rel(out[0][k], out[1][k]) < 1.5e-6
