"""Default tile of the hex Helmholtz kernels with per-point geometry: on both
sides of the line between the vector and the matrix-core tile, Q = NUMMODES
included, one element, odd counts, alone and in a batch.  Oracle and bounds as
for the tiles themselves (relative to the largest value, FP64 1e-12, FP32
2e-5); a member of a batch has to be what it is alone, bit for bit."""
import numpy as np
import pytest

import _oracle as O
import geometry_cases as G
import test_gpu_batch as B

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
nmf = B.nmf


@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nm,nq", [(5, 6), (6, 7), (6, 8), (7, 8), (8, 8), (7, 9), (8, 9), (8, 10), (9, 10),
                                   (10, 10), (9, 11), (10, 11), (10, 12)])
def test_default_tile(nmf, nm, nq, fp32):
    items = [B.Item(nmf, "Helmholtz", O.HEX, nm, nq, n, True, fp32, 0.3 + n, 40 + n) for n in (1, 5, 27)]
    ref = [it.alone()[0] for it in items]
    for it, y in zip(items, ref):
        want = O.helmholtz(O.HEX, nm, nq, it.nelmt, True, it.jac, it.df, it.lam, it.x_host)
        assert G.rel_err(y, want) <= (2e-5 if fp32 else 1e-12), it.nelmt
    if nq == nm:  # batches take Q = NUMMODES + 1 and + 2 only
        return
    b = nmf.Batch(mode=1)
    for it in items:
        it.reset()
        b.add(it.op, it.x, it.outs[0])
    b.run()
    torch.cuda.synchronize()
    for it, y in zip(items, ref):
        assert np.array_equal(it.got()[0], y), it.nelmt


def test_single_precision_line_in_elements(nmf):
    """FP32 at NQ = 11: matrix cores (tile TILE_MFMA + 1) as long as they need
    no more rounds over the card than the vector tile (2 elements); the two sum
    in other orders, so the bits tell which one ran."""
    nm, nq, nqt = 9, 11, 11 ** 3
    rng = np.random.default_rng(6)
    batch, alone = nmf.Batch(mode=nmf.Batch.GROUPED), []
    for nel, tile in ((1536, nmf.TILE_MFMA + 1), (1537, 2), (2048, 2), (2049, nmf.TILE_MFMA + 1)):
        op = nmf.GetOperatorFactory().CreateInstance("Helmholtz_Hex_Deformed", nm, nq, nel, nmf.FP32)
        op.SetJac(rng.uniform(0.5, 1.5, nel * nqt))
        op.SetDF(np.tile(np.eye(3).reshape(-1), nel * nqt) + rng.uniform(-0.2, 0.2, nel * nqt * 9))
        op.SetLambda(0.7)
        x = torch.from_numpy(rng.uniform(-1, 1, nel * nm ** 3)).float().cuda()
        got = {}
        for t in (0, nmf.TILE_MFMA + 1, 2):
            op.tile = t
            got[t] = torch.zeros_like(x)
            op(x, got[t])
        op.tile = 0
        torch.cuda.synchronize()
        assert not torch.equal(got[nmf.TILE_MFMA + 1], got[2])
        assert torch.equal(got[0], got[tile]), nel
        y = torch.zeros_like(x)
        batch.add(op, x, y)
        alone.append((got[0], y))
    assert batch.info()["groups"] == 2
    batch.run()
    torch.cuda.synchronize()
    for want, y in alone:
        assert torch.equal(want, y)
