"""Hex PhysDeriv on both sides of the line from which it runs in two LDS slabs
instead of three: as many elements as the card holds at once with three, and
one more (the line of Q = 4 back to three, in FP64, is crossed the same way).  The two forms do the same sums, so the common elements agree bit
for bit; the first and the last elements are held against the oracle
(relative to the largest value, FP64 1e-12, FP32 2e-5 as for the other
operators)."""
import numpy as np
import pytest

import _oracle as O

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def nmf():
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import nektar_amd
    nektar_amd.lib()
    return nektar_amd


def held_at_once(nq, fp32, slabs):
    """Elements resident on 256 CUs of 160 KB LDS and 32 waves."""
    per = max(1, 256 // nq ** 2)
    lds = per * slabs * nq * nq * (nq | 1) * (4 if fp32 else 8)
    return 256 * min(160 * 1024 // lds, 32 // ((per * nq * nq + 63) // 64)) * per


@pytest.mark.parametrize("nq,slabs", [(4, 3), (4, 2), (5, 3), (6, 3), (9, 3), (12, 3)])
@pytest.mark.parametrize("deformed", [False, True], ids=["regular", "deformed"])
@pytest.mark.parametrize("fp32", [False, True], ids=["fp64", "fp32"])
def test_same_sums_on_both_sides(nmf, nq, slabs, deformed, fp32):
    n, nqt, dt = held_at_once(nq, fp32, slabs), nq ** 3, torch.float32 if fp32 else torch.float64
    rng = np.random.default_rng(nq)
    df = np.tile(np.eye(3).reshape(-1), (n + 1) * (nqt if deformed else 1))
    df += 0.3 * rng.uniform(-1, 1, df.size)
    x = rng.uniform(-1, 1, (n + 1) * nqt)
    xd, per = torch.from_numpy(x).to(dt).cuda(), df.size // (n + 1)
    got = []
    for count in (n, n + 1):
        op = nmf.GetOperatorFactory().CreateInstance("PhysDeriv" + nmf.GetOpstring("Hex", deformed), nq - 1, nq, count,
                                                     nmf.FP32 if fp32 else nmf.FP64)
        op.SetDF(df[:count * per])
        y = [torch.full((count * nqt + 8,), 5.0, dtype=dt, device="cuda") for _ in range(3)]
        op(xd[:count * nqt], *[o[:count * nqt] for o in y])
        torch.cuda.synchronize()
        assert all(bool((o[count * nqt:] == 5.0).all()) for o in y)  # nothing past the last element
        got.append([o[:count * nqt].double().cpu().numpy() for o in y])
    for a, b in zip(*got):
        assert np.array_equal(a, b[:n * nqt])
    for e in (0, n):
        want = O.physderiv(O.HEX, nq - 1, nq, 1, deformed, df[e * per:(e + 1) * per], x[e * nqt:(e + 1) * nqt])
        scale = max(np.max(np.abs(w)) for w in want)
        for g, w in zip(got[1], want):
            assert np.max(np.abs(g[e * nqt:(e + 1) * nqt] - w)) <= (2e-5 if fp32 else 1e-12) * scale
