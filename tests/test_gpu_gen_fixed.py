"""Prism and pyramid kernels with compile-time sizes: every compiled NUMMODES
with Q = NUMMODES + 1 and + 2, every operator, and more elements than
workgroups of the walking grid (4096).  Oracle and bounds as for the
runtime-size operators (relative to the largest value, FP64 1e-12, FP32 5e-5):
the stages and the order of their sums are the same."""
import numpy as np
import pytest

import _oracle as O
import geometry_cases as G
import test_gpu_runtime_size as R

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
nmf = R.nmf

SIZES = [(nm, nm + d, 11) for nm in range(3, 8) for d in (1, 2)] + [(3, 4, 4099)]


@pytest.mark.parametrize("shape", ["Prism", "Pyr"])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("deformed", [False, True], ids=["regular", "deformed"])
def test_every_size_and_operator(nmf, shape, prec, deformed):
    P, geo = (nmf.FP64 if prec == "fp64" else nmf.FP32), "Deformed" if deformed else "Regular"
    S = O.PRISM if shape == "Prism" else O.PYR
    for ci, (n, q, E) in enumerate(SIZES):
        nm, nq = (n, n, n), (q, q, q - 1)
        nqt, nc = int(np.prod(nq)), O.ncoeffs_aniso(S, nm)
        jac, df = R._geom(E, nqt, deformed, 500 + ci)
        x = G.coeffs(E * nc, 600 + ci)
        f = [G.coeffs(E * nqt, 700 + 3 * ci + k) for k in range(3)]
        vel = np.random.default_rng(800 + ci).uniform(-1.0, 1.0, E * nqt * 3)
        u = O.bwdtrans_aniso(S, nm, nq, E, x)
        runs = [("BwdTrans", [x], [E * nqt], {}, [u]),
                ("IProduct", [f[0]], [E * nc], {}, [O.iproduct_aniso(S, nm, nq, E, deformed, jac, f[0])]),
                ("PhysDeriv", [u], [E * nqt] * 3, {}, list(O.physderiv_aniso(S, nm, nq, E, deformed, df, u))),
                ("IProductWRTDerivBase", f, [E * nc], {}, [O.iproduct_deriv_aniso(S, nm, nq, E, deformed, jac, df, *f)]),
                ("Helmholtz", [x], [E * nc], {"lam": 0.7},
                 [O.helmholtz_aniso(S, nm, nq, E, deformed, jac, df, 0.7, x, None)]),
                ("LinearAdvectionDiffusionReaction", [x], [E * nc], {"lam": 1.3, "vel": vel},
                 [O.adv_diff_react_aniso(S, nm, nq, E, deformed, jac, df, vel, 1.3, x)])]
        for op, ins, outs, kw, want in runs:
            tag = "Regular" if op == "BwdTrans" else geo
            got = R._run(nmf, f"{op}_{shape}_{tag}", nm, nq, E, P, jac, df, ins, outs, **kw)
            R._check(got, want, P, nmf, (shape, nm, nq, E, prec, geo, op))
