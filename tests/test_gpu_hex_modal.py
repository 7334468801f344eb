"""Legendre-space Helmholtz kernels of affine hexahedra (constant Jacobian
and metric per element), where they can go wrong: every compiled NUMMODES,
points Q = NUMMODES (the top Legendre norm is the rule's, not the exact
one), + 1 and + 2, element counts around a workgroup's, a full diffusion
tensor and sheared elements (every mixed metric term).

The reference sums over the points what these kernels sum in 1-D: the same
numbers up to rounding, so the bounds are those of the other operator tests,
relative to the largest value: FP64 1e-12, FP32 2e-5."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DIFF6 = [1.3, 0.2, 0.9, -0.1, 0.15, 1.7]


@pytest.fixture(scope="module")
def nmf():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import nektar_amd
    nektar_amd.lib()
    return nektar_amd


def sheared(nel, seed):
    rng = np.random.default_rng(seed)
    M = 0.1 * (np.eye(3)[None] + 0.3 * rng.uniform(-1, 1, (nel, 3, 3)))
    return np.abs(np.linalg.det(M)), np.transpose(np.linalg.inv(M), (0, 2, 1)).reshape(-1)


@pytest.mark.parametrize("nm,nq", [(2, 3), (2, 4)] + [(nm, nm + d) for nm in range(3, 11) for d in (0, 1, 2)])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_against_oracle_around_a_workgroup(nmf, nm, nq, fp32):
    per = 64 // nm ** 2 if nm <= 4 else 5 if nm <= 6 else 2 if nm == 9 else 1
    dt = torch.float32 if fp32 else torch.float64
    for nel, diff6 in ((1, None), (per + 1, DIFF6), (3 * per, None)):
        jac, df = sheared(nel, 10 * nm + nel)
        op = nmf.GetOperatorFactory().CreateInstance("Helmholtz_Hex_Regular", nm, nq, nel,
                                                     nmf.FP32 if fp32 else nmf.FP64)
        op.SetJac(jac)
        op.SetDF(df)
        op.SetLambda(0.7)
        op.SetConstVarDiffusion(diff6)
        x = O.splitmix_uniform(nel, nel * nm ** 3)
        guard = 8  # nothing is written past the last element
        y = torch.full((nel * nm ** 3 + guard,), 5.0, dtype=dt, device="cuda")
        op(torch.from_numpy(x).to(dt).cuda(), y[:nel * nm ** 3])
        torch.cuda.synchronize()
        got = y.double().cpu().numpy()
        assert np.all(got[nel * nm ** 3:] == 5.0)
        ref = O.helmholtz(O.HEX, nm, nq, nel, False, jac, df, 0.7, x, diff6)
        err = np.max(np.abs(got[:nel * nm ** 3] - ref)) / np.max(np.abs(ref))
        assert err <= (2e-5 if fp32 else 1e-12), (nel, err)


@pytest.mark.parametrize("nm,nq", [(nm, nm + d) for nm in range(2, 11) for d in (1, 2)])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_default_tile_is_a_candidate(nmf, nm, nq, fp32):
    """The autotuner can choose the default's elements per workgroup, alone and
    in a batch, and gets the default's results."""
    per = 64 // nm ** 2 if nm <= 4 else 5 if nm <= 6 else 2 if nm == 9 else 1
    nel, dt = 2 * per + 1, torch.float32 if fp32 else torch.float64
    jac, df = sheared(nel, nm)
    op = nmf.GetOperatorFactory().CreateInstance("Helmholtz_Hex_Regular", nm, nq, nel, nmf.FP32 if fp32 else nmf.FP64)
    op.SetJac(jac)
    op.SetDF(df)
    op.SetLambda(0.7)
    assert op.tile == 0 and per in op.tile_candidates()
    x = torch.from_numpy(O.splitmix_uniform(nel, nel * nm ** 3)).to(dt).cuda()
    default, pinned, grouped = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x)
    op(x, default)
    op.tile = per
    op(x, pinned)
    batch = nmf.Batch(mode=nmf.Batch.GROUPED)
    batch.add(op, x, grouped)
    batch.run()
    torch.cuda.synchronize()
    assert torch.equal(default, pinned) and torch.equal(default, grouped)
