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
