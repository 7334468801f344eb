"""The structured solver's CG iteration in three launches (assembly fused with
the vector updates, s.w as one dot per element): every compiled NUMMODES,
meshes whose grid lines do not fill the 64- and 128-row pieces of a wave or
whose line count does not divide among the XCDs, the smallest mesh, affine and
perturbed elements.

The dots only steer the iteration, so a wrong one shows as a residual that the
recurrence does not know of: the true residual b - A x, taken with
apply_global (assembled by another kernel), has to be what the solve reports.
The recurrence residual is below 1e-10 ||b||; rounding of some hundred updates
of a system of condition below 1e6 adds less than 1e-9 ||b||."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def nmf():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import nektar_amd
    nektar_amd.lib()
    return nektar_amd


def check_true_residual(s, n, nm, mixed=False):
    s.set_forcing_manufactured(1)
    info = s.solve(mixed, tol=1e-10, maxit=8000)
    assert info.converged, (n, info.as_dict())
    x = torch.from_numpy(s.solution()).cuda()
    y = torch.zeros_like(x)
    s.apply_global(x, y)
    torch.cuda.synchronize()
    b, N = s.rhs().reshape((n * (nm - 1) + 1,) * 3), n * (nm - 1) + 1
    res = (b - y.cpu().numpy().reshape(b.shape))[1:N - 1, 1:N - 1, 1:N - 1]
    assert np.linalg.norm(res) <= 1.1e-9 * np.linalg.norm(b), (n, np.linalg.norm(res) / np.linalg.norm(b))


@pytest.mark.parametrize("nm", range(2, 11))
@pytest.mark.parametrize("perturb", [0.0, 0.1], ids=["affine", "perturbed"])
def test_true_residual(nmf, nm, perturb):
    for n in (2, 3, 13 if nm == 6 else 7 if nm < 9 else 4):
        check_true_residual(nmf.HelmholtzSolver(n, nm, nm + 1, 1.3, perturb=perturb, seed=3), n, nm)


@pytest.mark.parametrize("n", [32, 33])
@pytest.mark.parametrize("perturb", [0.0, 0.1], ids=["affine", "perturbed"])
def test_true_residual_around_the_direct_sum(nmf, n, perturb):
    """Up to 32^3 elements the scalar step adds the element dots itself, above
    it adds their sums by workgroup."""
    check_true_residual(nmf.HelmholtzSolver(n, 2, 3, 1.3, perturb=perturb, seed=3), n, 2)


@pytest.mark.parametrize("nm,d", [(2, 1), (2, 2), (3, 1), (4, 2), (5, 1), (5, 2), (6, 2), (7, 1), (8, 2), (9, 1), (10, 1),
                                  (10, 2)])
@pytest.mark.parametrize("perturb", [0.0, 0.1], ids=["affine", "perturbed"])
def test_true_residual_of_every_tile(nmf, nm, d, perturb):
    """Every producer of the element dots: the gather kernels at each tile, and
    the separate dot after a matrix-core tile.  The vector tiles do the same
    sums, so their iterates agree bit for bit, and so do the matrix-core ones."""
    key = "Helmholtz" + nmf.GetOpstring("Hex", perturb != 0.0)
    cand = [nmf.GetOperatorFactory().CreateInstance(key, nm, nm + d, 1, p).tile_candidates()
            for p in (nmf.FP64, nmf.FP32)]
    for n in (1, 3) if nm > 2 else (2, 5):
        s = nmf.HelmholtzSolver(n, nm, nm + d, 1.3, perturb=perturb, seed=3)
        solutions = {}
        for tile in [0] + cand[0]:
            s.set_tiles(tile, 0)
            check_true_residual(s, n, nm)
            same = solutions.setdefault(tile >= nmf.TILE_MFMA, s.solution())
            assert np.array_equal(same, s.solution()), tile
        for tile in cand[1]:
            s.set_tiles(0, tile)
            check_true_residual(s, n, nm, mixed=True)
        with pytest.raises(nmf.NektarError):
            s.set_tiles(3 if nm not in (9, 10) else 5, 0)


@pytest.mark.parametrize("n,nm,mixed", [(35, 5, True), (36, 5, True), (44, 5, False), (45, 5, False)])
def test_true_residual_around_the_cache(nmf, n, nm, mixed):
    """Perturbed elements whose per-point geometry (7 values per point) is just
    below and just above the 256 MB (FP32) and 1 GB (FP64) from which the
    gather deals its workgroups to the XCDs in another order."""
    size = n ** 3 * 7 * (nm + 1) ** 3 * (4 if mixed else 8) / 2 ** 20
    assert (size > (256 if mixed else 1024)) == (n in (36, 45))
    check_true_residual(nmf.HelmholtzSolver(n, nm, nm + 1, 1.3, perturb=0.1, seed=3), n, nm, mixed)
