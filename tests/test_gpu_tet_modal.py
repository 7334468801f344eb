"""Matrix-core Helmholtz kernels of affine tetrahedra where they can go wrong:
every compiled NUMMODES (the matrices are cut into 16x4 blocks by it), element
counts around 16 and 64 (a wave's and a workgroup's) and around the count from
which a wave keeps its elements to itself, a full diffusion tensor, and both
variants side by side in one grouped launch.

The products are those of the reference up to the order of their sums, so the
bounds are those of the other operator tests, relative to the largest value:
FP64 1e-12, FP32 2e-5 (2e-4 above 7 modes)."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

DIFF6 = [1.3, 0.2, 0.9, -0.1, 0.15, 1.7]
SPLIT = 640 * 16  # up to here four waves share 16 elements


@pytest.fixture(scope="module")
def nmf():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import nektar_amd
    nektar_amd.lib()
    return nektar_amd


def sheared(nel, seed):
    rng = np.random.default_rng(seed)
    M = 0.05 * (np.eye(3)[None] + 0.3 * rng.uniform(-1, 1, (nel, 3, 3)))
    return np.abs(np.linalg.det(M)), np.transpose(np.linalg.inv(M), (0, 2, 1)).reshape(-1)


def operator(nmf, nm, nq, nel, fp32, diff6):
    jac, df = sheared(nel, 10 * nm + nel % 7)
    op = nmf.GetOperatorFactory().CreateInstance("Helmholtz_Tet_Regular", nm, nq, nel, nmf.FP32 if fp32 else nmf.FP64)
    op.SetJac(jac)
    op.SetDF(df)
    op.SetLambda(0.7)
    op.SetConstVarDiffusion(diff6)
    return op, jac, df


def check(got, nm, nq, nel, jac, df, x, diff6, fp32):
    ref = O.helmholtz(O.TET, nm, nq, nel, False, jac, df, 0.7, x, diff6)
    err = np.max(np.abs(got - ref)) / np.max(np.abs(ref))
    assert err <= ((2e-5 if nm <= 7 else 2e-4) if fp32 else 1e-12), (nm, nel, err)


@pytest.mark.parametrize("nm", range(2, 11))
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_against_oracle_around_a_wave(nmf, nm, fp32):
    dt = torch.float32 if fp32 else torch.float64
    nc = nm * (nm + 1) * (nm + 2) // 6
    for nel, nq, diff6 in ((1, nm + 1, None), (17, nm + 2, DIFF6), (64, nm + 1, None)):
        op, jac, df = operator(nmf, nm, nq, nel, fp32, diff6)
        x = O.splitmix_uniform(nel, nel * nc)
        y = torch.full((nel * nc + 8,), 5.0, dtype=dt, device="cuda")  # nothing is written past the end
        op(torch.from_numpy(x).to(dt).cuda(), y[:nel * nc])
        torch.cuda.synchronize()
        got = y.double().cpu().numpy()
        assert np.all(got[nel * nc:] == 5.0)
        check(got[:nel * nc], nm, nq, nel, jac, df, x, diff6, fp32)


@pytest.mark.parametrize("nm", [3, 6])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_both_variants_alone_and_grouped(nmf, nm, fp32):
    dt = torch.float32 if fp32 else torch.float64
    nc = nm * (nm + 1) * (nm + 2) // 6
    batch = nmf.Batch(mode=nmf.Batch.GROUPED, streams=1)
    outs = []
    for nel in (SPLIT, SPLIT + 1, 33, SPLIT + 47):
        op, jac, df = operator(nmf, nm, nm + 1, nel, fp32, None)
        x = O.splitmix_uniform(nel, nel * nc)
        xd, y = torch.from_numpy(x).to(dt).cuda(), torch.zeros(nel * nc, dtype=dt, device="cuda")
        grouped = torch.zeros_like(y)
        op(xd, y)
        batch.add(op, xd, grouped)
        outs.append((y, grouped))
        torch.cuda.synchronize()
        check(y.double().cpu().numpy(), nm, nm + 1, nel, jac, df, x, None, fp32)
    batch.run()
    torch.cuda.synchronize()
    for y, grouped in outs:
        assert torch.equal(y, grouped)


def test_one_group_whatever_the_tile(nmf):
    """One kernel serves every tile of affine tets, so members with different
    tiles share a launch."""
    batch = nmf.Batch(mode=nmf.Batch.GROUPED)
    outs = []
    for k, nel in enumerate((5, 70, 33)):
        op, _, _ = operator(nmf, 4, 5, nel, False, None)
        op.tile = ([0] + op.tile_candidates())[k]
        x = torch.from_numpy(O.splitmix_uniform(nel, nel * 20)).cuda()
        y, grouped = torch.zeros_like(x), torch.zeros_like(x)
        op(x, y)
        batch.add(op, x, grouped)
        outs.append((y, grouped))
    assert batch.info()["groups"] == 1
    batch.run()
    torch.cuda.synchronize()
    for y, grouped in outs:
        assert torch.equal(y, grouped)
