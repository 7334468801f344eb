"""Performance cases of the matrix-free operators and the solves built on them.

Every case is one pass that a program using this package makes: a Helmholtz
apply inside somebody's Krylov loop, an explicit right-hand side, an uneven
batch of collections, one solve.  ``listed()`` names the fixed ones,
``draw(rng)`` gives others of the same ranges.

A case is a dict with

    kind   "helmholtz"  y = (lambda M + L) x on one collection of elements
           "advection"  the same with an advection velocity per point
           "explicit"   BwdTrans, PhysDeriv, IProductWRTDerivBase, IProduct:
                        the calls of an explicit time step
           "batch"      a batch of Helmholtz collections, hex and tet, uneven
           "solve"      preconditioned CG on a structured hex mesh
    shape  "Hex" | "Tet" | "Prism"
    nm     modes per direction (polynomial order + 1)
    nq     points in direction 0
    E      elements
    curved per-point geometry instead of one Jacobian per element
    single FP32 instead of FP64
    tuned  the program calls autotune() once at set-up
"""
import math

import numpy as np
import torch

import nektar_amd

MODES = (3, 10)       # modes per direction: orders 2 .. 9
LARGEST_DOFS = 11.3e6  # the 32^3 mesh at order 6
KEYS = {"kind": "helmholtz", "shape": "Hex", "nm": 7, "nq": 8, "E": 1, "curved": False, "single": False,
        "tuned": False}


def _case(name=None, **kw):
    c = dict(KEYS)
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest call: a coarse mesh, where launch latency is all there is
        _case("hex_p4_64", nm=5, nq=6, E=64),
        # the 32^3 mesh at order 6, the benchmark's apply (which tunes once at set-up)
        _case("hex_p6_32cubed", nm=7, nq=8, E=32768, tuned=True),
        # a low-order FP32 apply of a mixed-precision iteration, over-integrated, ragged count
        _case("hex_p3_single", nm=4, nq=6, E=50021, single=True),
        # curved elements, order 7: per-point geometry
        _case("hex_p7_curved", nm=8, nq=9, E=2197, curved=True),
        # an unstructured tet mesh at order 6
        _case("tet_p6_32768", shape="Tet", nm=7, nq=8, E=32768, tuned=True),
        # high-order tets in FP32, ragged count
        _case("tet_p9_single", shape="Tet", nm=10, nq=11, E=4001, single=True),
        # curved tets of a boundary layer
        _case("tet_p4_curved", shape="Tet", nm=5, nq=6, E=3001, curved=True),
        # boundary-layer prisms
        _case("prism_p4", shape="Prism", nm=5, nq=6, E=4096),
        # one explicit right-hand side (transform, gradient, weak forms) on hexes
        _case("hex_p5_explicit", kind="explicit", nm=6, nq=7, E=8192),
        # advection-diffusion-reaction on tets, a velocity per point
        _case("tet_p5_advection", kind="advection", shape="Tet", nm=6, nq=7, E=6007),
        # a mesh of many collections: hex and tet, orders 3 to 9, applied as one submission
        _case("batch_16", kind="batch", E=6000, items=16, tuned=True),
        # one Helmholtz solve on the unit box to 1e-10
        _case("solve_16cubed", kind="solve", nm=7, nq=8, n=16, E=4096, perturb=0.0),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["helmholtz"] * 6 + ["explicit", "explicit", "advection", "advection", "batch", "solve"])
    if kind == "batch":
        return _case(kind=kind, E=_logint(rng, 500, 6000), items=rng.randint(3, 16), tuned=rng.random() < 0.5,
                     single=rng.random() < 0.35)
    if kind == "solve":
        nm = rng.randint(3, 8)
        perturb = rng.choice([0.0, 0.0, 0.1])
        # a perturbed mesh takes more iterations, each with geometry per point
        n = rng.randint(3, 6 if perturb else max(3, min(16, 96 // (nm - 1))))
        return _case(kind=kind, nm=nm, nq=nm + rng.randint(1, 2), n=n, E=n ** 3, perturb=perturb)
    shape = rng.choice(["Hex"] * 4 + ["Tet"] * 4 + (["Prism"] if kind == "helmholtz" else []))
    nm = rng.randint(*MODES)
    if shape == "Prism":
        nm = rng.randint(3, 6)
    nq = nm + rng.choice([1, 1, 2])
    curved = rng.random() < 0.3
    # work in points x modes: at most the 32^3 mesh; curved, advected and
    # explicit collections carry data per point, prisms run at runtime size
    points = nq ** 3 if shape == "Hex" else nq * nq * (nq - 1) if shape == "Prism" else nq * (nq - 1) ** 2
    heavy = curved or kind != "helmholtz" or shape == "Prism"
    most = max(64, int(min(50000, (1.4e6 if heavy else 0.9 * LARGEST_DOFS) / points)))
    return _case(kind=kind, shape=shape, nm=nm, nq=nq, E=_logint(rng, 20, most), curved=curved,
                 single=rng.random() < 0.35)


# ------------------------------------------------------------ sizes
def _ncoeff(shape, nm):
    if shape == "Hex":
        return nm ** 3
    if shape == "Tet":
        return nm * (nm + 1) * (nm + 2) // 6
    return nm * nm * (nm + 1) // 2


def _points(shape, nq):
    if shape == "Hex":
        return nq ** 3
    if shape == "Tet":
        return nq * (nq - 1) ** 2
    return nq * nq * (nq - 1)


def _batch_items(case):
    """(shape, nm, E) of the batch's collections, from the case alone: hex and
    tet alternating, orders 3..9, counts from a sixth of E to E."""
    out = []
    for i in range(case["items"]):
        nm = 4 + (5 * i + case["items"]) % 7
        out.append(("Hex" if i % 2 == 0 else "Tet", nm, max(1, int(case["E"] * (1 + (7 * i) % 11) / 11))))
    return out


def _sum_factorised(shape, nm, nq):
    """Flops of one Helmholtz element by sum factorisation at the points:
    transforms there and back, collocation gradient and its transpose, metric."""
    if shape == "Hex":
        T = 2 * (nm ** 3 * nq + nm ** 2 * nq ** 2 + nm * nq ** 3)
        return 2 * T + 12 * nq ** 4 + 18 * nq ** 3
    pts = _points(shape, nq)
    if shape == "Tet":
        q1 = nq - 1
        T = 2 * (q1 * _ncoeff(shape, nm) + q1 * q1 * nm * (nm + 1) // 2 + pts * nm)
        return 2 * T + 4 * pts * (nq + 2 * q1) + 30 * pts
    q2 = nq - 1
    T = 2 * (q2 * _ncoeff(shape, nm) + q2 * nq * nm * nm + pts * nm)
    return 2 * T + 4 * pts * (2 * nq + q2) + 30 * pts


def _helmholtz_work(shape, nm, nq, E, curved, size, advected=False):
    """Bytes and flops of one Helmholtz-type apply.  With constant geometry
    the element matrix is a sum of seven fixed ones: on a hex each is a
    product of 1-D matrices with a few bands (some 70 flops per coefficient),
    on a tet gradients into the polynomials one degree lower, half of their
    entries zero by the reflection of the reference element."""
    nc, pts = _ncoeff(shape, nm), _points(shape, nq)
    geo = (7 if shape == "Hex" else 10) * (pts if curved else 1)
    flops = _sum_factorised(shape, nm, nq)
    if not curved and not advected:
        if shape == "Hex":
            flops = min(flops, 70 * nc)
        elif shape == "Tet":
            lower = _ncoeff(shape, nm - 1)
            flops = min(flops, nc * (6 * lower + nc))
    byts = (2 * nc + geo + (3 * pts if advected else 0)) * size
    return {"bytes": E * byts, "flops": E * flops}


def work(case):
    size = 4 if case["single"] else 8
    if case["kind"] == "batch":
        w = [_helmholtz_work(s, nm, nm + 1, E, False, size) for s, nm, E in _batch_items(case)]
        return {k: sum(x[k] for x in w) for k in ("bytes", "flops")}
    nm, nq, E, shape = case["nm"], case["nq"], case["E"], case["shape"]
    if case["kind"] == "solve":
        # the Jacobi-preconditioned iterations grow with the order: about 100 for each
        # (a third more on a perturbed mesh); each reads and writes the solution,
        # residual and direction, and applies the operator
        its = (130 if case["perturb"] else 100) * (nm - 1)
        rows = (case["n"] * (nm - 1) + 1) ** 3
        w = _helmholtz_work("Hex", nm, nq, E, case["perturb"] != 0, 8)
        return {"bytes": its * (w["bytes"] + 6 * 8 * rows), "flops": its * (w["flops"] + 12 * rows)}
    if case["kind"] == "explicit":
        nc, pts = _ncoeff(shape, nm), _points(shape, nq)
        geo = 10 * (pts if case["curved"] else 1)
        transform = _sum_factorised(shape, nm, nq) / 4
        return {"bytes": E * size * (3 * nc + 9 * pts + 3 * geo), "flops": int(E * 4 * transform)}
    return _helmholtz_work(shape, nm, nq, E, case["curved"], size, case["kind"] == "advection")


# ------------------------------------------------------------ inputs
def _geometry(case, shape, nq, E, curved, seed):
    """Jacobian and inverse map derivatives of sheared elements of size ~0.1
    (curved: with a smooth variation over the element), as a mesh reader
    hands them over: host arrays per element, or per point."""
    rng = np.random.default_rng(seed)
    h = rng.uniform(0.5, 2.0, E)[:, None, None] * (0.05 if shape == "Hex" else 0.025)
    M = h * (np.eye(3)[None] + 0.25 * rng.uniform(-1, 1, (E, 3, 3)))
    if not curved:
        jac = np.abs(np.linalg.det(M))
        return jac, np.ascontiguousarray(np.transpose(np.linalg.inv(M), (0, 2, 1))).reshape(-1)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    z = [torch.from_numpy(_rule(shape, d, nq)[0]).to(dev) for d in range(3)]
    pts = [z[0][None, None, :], z[1][None, :, None], z[2][:, None, None]]
    amp = torch.from_numpy(0.15 * rng.uniform(-1, 1, (E, 3, 3, 1, 1, 1))).to(dev)
    Mt = torch.from_numpy(M)[..., None, None, None].to(dev)
    wave = torch.stack([torch.cos(1.3 * pts[0] + 0.4 * pts[1]) + 0 * pts[2],
                        torch.cos(1.1 * pts[1] - 0.5 * pts[2]) + 0 * pts[0],
                        torch.cos(0.9 * pts[2] + 0.3 * pts[0]) + 0 * pts[1]])
    A = (Mt * (1 + amp * wave[None, None])).permute(0, 3, 4, 5, 1, 2).reshape(-1, 3, 3)
    det = torch.linalg.det(A)
    inv = torch.linalg.inv(A).transpose(1, 2).contiguous()
    return det.abs().cpu().numpy(), inv.reshape(-1).cpu().numpy()


def _values(n, single, seed):
    """Coefficients or point values in [-1, 1)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    g = torch.Generator(device=dev).manual_seed(seed)
    dt = torch.float32 if single else torch.float64
    return torch.rand(n, dtype=dt, device=dev, generator=g) * 2 - 1


def _forcing(case, seed):
    """A smooth source on the unit box at the quadrature points: a few
    standing waves and a Gaussian bump."""
    n, nq = case["n"], case["nq"]
    rng = np.random.default_rng(seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x1 = (np.arange(n)[:, None] + 0.5 * (1 + _rule("Hex", 0, nq)[0])) / n  # [element, point] of a line
    x = [torch.from_numpy(x1).to(dev).reshape([n if i == a else nq if i == a + 3 else 1 for i in range(6)])
         for a in (2, 1, 0)]  # axes: element z, y, x, point z, y, x
    f = 0
    for _ in range(4):
        k, a = rng.integers(1, 4, 3), rng.uniform(-1, 1)
        f = f + a * torch.sin(math.pi * int(k[0]) * x[0]) * torch.sin(math.pi * int(k[1]) * x[1]) * torch.sin(
            math.pi * int(k[2]) * x[2])
    c = rng.uniform(0.3, 0.7, 3)
    f = f + torch.exp(-40 * sum((x[d] - float(c[d])) ** 2 for d in range(3)))
    return f.contiguous().reshape(-1)


def _operator(name, shape, case, nq, nm, E, jac, df, lam=None, velocity=None):
    key = name + nektar_amd.GetOpstring(shape, case["curved"])
    op = nektar_amd.GetOperatorFactory().CreateInstance(
        key, nm, nq, E, nektar_amd.FP32 if case["single"] else nektar_amd.FP64)
    if name not in ("BwdTrans", "PhysDeriv"):
        op.SetJac(jac)
    if name not in ("BwdTrans", "IProduct"):
        op.SetDF(df)
    if lam is not None:
        op.SetLambda(lam)
    if velocity is not None:
        op.SetAdvectionVelocities(velocity)
    if case["tuned"] and case["kind"] != "batch":
        op.autotune()
    return op


def _empty(n, single):
    return torch.empty(n, dtype=torch.float32 if single else torch.float64, device="cuda")


def _lambda(seed):
    return 0.5 + (seed % 17) / 8.0


def _velocity(case, seed):
    rng = np.random.default_rng(seed + 77)
    return rng.uniform(-1, 1, 3 * case["E"] * _points(case["shape"], case["nq"]))


def prepare(case, seed):
    nm, nq, E, shape, single = case["nm"], case["nq"], case["E"], case["shape"], case["single"]
    if case["kind"] == "solve":
        s = nektar_amd.HelmholtzSolver(case["n"], nm, nq, _lambda(seed), perturb=case["perturb"], seed=seed)
        s.set_forcing_phys(_forcing(case, seed))
        return {"kind": "solve", "solver": s}
    if case["kind"] == "batch":
        b = nektar_amd.Batch()
        outs = []
        for i, (sh, m, e) in enumerate(_batch_items(case)):
            jac, df = _geometry(case, sh, m + 1, e, False, seed + 1000 * i)
            op = _operator("Helmholtz", sh, case, m + 1, m, e, jac, df, _lambda(seed + i))
            x = _values(op.input_size(), single, seed + 1000 * i)
            y = _empty(op.output_size(), single)
            b.add(op, x, y)
            outs.append(y)
        if case["tuned"]:
            b.autotune()
        return {"kind": "batch", "batch": b, "outs": outs}
    jac, df = _geometry(case, shape, nq, E, case["curved"], seed)
    nc, pts = E * _ncoeff(shape, nm), E * _points(shape, nq)
    x = _values(nc, single, seed)
    if case["kind"] == "explicit":
        ops = [_operator(n, shape, case, nq, nm, E, jac, df)
               for n in ("BwdTrans", "PhysDeriv", "IProductWRTDerivBase", "IProduct")]
        bufs = [_empty(pts, single) for _ in range(4)] + [_empty(nc, single) for _ in range(2)]
        return {"kind": "explicit", "ops": ops, "x": x, "bufs": bufs}
    if case["kind"] == "advection":
        op = _operator("LinearAdvectionDiffusionReaction", shape, case, nq, nm, E, jac, df, _lambda(seed),
                       _velocity(case, seed))
    else:
        op = _operator("Helmholtz", shape, case, nq, nm, E, jac, df, _lambda(seed))
    return {"kind": "apply", "op": op, "x": x, "y": _empty(nc, single)}


def run(state):
    if state["kind"] == "apply":
        state["op"](state["x"], state["y"])
        return state["y"]
    if state["kind"] == "explicit":
        bwd, grad, weak, mass = state["ops"]
        u, d0, d1, d2, y, m = state["bufs"]
        bwd(state["x"], u)
        grad(u, d0, d1, d2)
        weak((d0, d1, d2), y)
        mass(u, m)
        return [u, d0, d1, d2, y, m]
    if state["kind"] == "batch":
        state["batch"].run()
        return state["outs"]
    state["solver"].solve(tol=1e-10)
    return state["solver"].solution()


def tolerance(case):
    # about four times the distance of the kernels from exact() below, over
    # some hundred and thirty cases of these ranges
    if case["kind"] == "solve":
        # solves that stop at a relative residual of 1e-10: up to 1e-6 from
        # one that goes on to 1e-13
        return {"rel": 4e-6, "max": 1e-4}
    single = case["single"]
    if case["kind"] == "explicit" and case["shape"] == "Tet":
        # nodal derivatives next to the collapsed vertex: rounding of the
        # point values times 4 / ((1 - b)(1 - c)), the more points the more
        return {"rel": 1.6e-4, "max": 1e-2} if single else {"rel": 4e-13, "max": 4e-11}
    return {"rel": 4e-6, "max": 8e-5} if single else {"rel": 1.2e-14, "max": 2e-13}


# ------------------------------------------------------------ 64-bit evaluation
def _jacobi(n, a, b, z):
    """P_n^{a,b}(z) and its derivative, three-term recurrence."""
    def val(n, a, b):
        if n < 0:
            return np.zeros_like(z)
        p0, p1 = np.ones_like(z), 0.5 * (a - b + (a + b + 2) * z)
        if n == 0:
            return p0
        for k in range(1, n):
            c = 2 * k + a + b
            p0, p1 = p1, (((c + 1) * (c * (c + 2) * z + a * a - b * b)) * p1
                          - 2 * (k + a) * (k + b) * (c + 2) * p0) / (2 * (k + 1) * (k + a + b + 1) * c)
        return p1
    return val(n, a, b), 0.5 * (n + a + b + 1) * val(n - 1, a + 1, b + 1)


def _roots(n, a, b):
    """Zeros of P_n^{a,b}: eigenvalues of the Jacobi matrix, then Newton."""
    if n == 0:
        return np.zeros(0)
    k = np.arange(n, dtype=float)
    s = 2 * k + a + b
    with np.errstate(divide="ignore", invalid="ignore"):
        d = (b * b - a * a) / (s * (s + 2))
    if a + b == 0:
        d[0] = (b - a) / (a + b + 2)
    k, s = k[1:], s[1:]
    e = np.sqrt(4 * k * (k + a) * (k + b) * (k + a + b) / (s ** 2 * (s + 1) * (s - 1)))
    if n > 1:
        e[0] = math.sqrt(4 * (1 + a) * (1 + b) / ((2 + a + b) ** 2 * (3 + a + b)))
    z = np.linalg.eigvalsh(np.diag(d) + np.diag(e, 1) + np.diag(e, -1))
    for _ in range(3):
        p, dp = _jacobi(n, a, b, z)
        z = z - p / dp
    return z


def _rule(shape, d, nq):
    """Points and weights of direction d: Gauss-Lobatto-Legendre, and in the
    collapsed directions Gauss-Radau-Jacobi at -1 for (1-z)^alpha, with the
    collapse's factor 2^-alpha in the weights."""
    alpha = {"Hex": (0, 0, 0), "Tet": (0, 1, 2), "Prism": (0, 0, 1)}[shape][d]
    if alpha == 0:
        z = np.concatenate([[-1.0], _roots(nq - 2, 1, 1), [1.0]])
        return z, 2.0 / (nq * (nq - 1) * _jacobi(nq - 1, 0, 0, z)[0] ** 2)
    n = nq - 1
    z = np.concatenate([[-1.0], _roots(n - 1, alpha, 1)])
    # exact for P_k^{alpha,0}, k < n, whose integrals against the weight vanish for k > 0
    V = np.stack([_jacobi(k, alpha, 0, z)[0] for k in range(n)])
    rhs = np.zeros(n)
    rhs[0] = 2.0 ** (alpha + 1) / (alpha + 1)
    return z, np.linalg.solve(V, rhs) * 0.5 ** alpha


def _mod_a(p, z):
    lo, hi = 0.5 * (1 - z), 0.5 * (1 + z)
    half = np.full_like(z, 0.5)
    if p < 2:
        return (lo, -half) if p == 0 else (hi, half)
    v, d = _jacobi(p - 2, 1, 1, z)
    return lo * hi * v, -0.5 * z * v + lo * hi * d


def _mod_b(p, q, z):
    lo, hi = 0.5 * (1 - z), 0.5 * (1 + z)
    if p == 0:
        return _mod_a(q, z)
    pw, dpw = lo ** p, -0.5 * p * lo ** (p - 1)
    if q == 0:
        return pw, dpw
    v, d = _jacobi(q - 1, 2 * p - 1, 1, z)
    return pw * hi * v, dpw * hi * v + pw * (0.5 * v + hi * d)


def _dense(shape, nm, nq):
    """Basis values [point, mode], standard-coordinate gradients [3, point,
    mode] and weights at the operator's points (direction 0 fastest)."""
    z, w = zip(*(_rule(shape, d, nq) for d in range(3)))
    c, b, a = (t.ravel() for t in np.meshgrid(z[2], z[1], z[0], indexing="ij"))
    W = (w[2][:, None, None] * w[1][None, :, None] * w[0][None, None, :]).ravel()
    one, half_p = (np.ones_like(a), np.zeros_like(a)), lambda t: (0.5 * (1 + t), np.full_like(t, 0.5))
    terms = []
    if shape == "Hex":
        for r in range(nm):
            for q in range(nm):
                for p in range(nm):
                    terms.append([(_mod_a(p, a), _mod_a(q, b), _mod_a(r, c))])
    elif shape == "Prism":
        for p in range(nm):
            for q in range(nm):
                for r in range(nm - p):
                    edge = p == 0 and r == 1
                    terms.append([(one, _mod_a(q, b), half_p(c)) if edge
                                  else (_mod_a(p, a), _mod_a(q, b), _mod_b(p, r, c))])
    else:
        for p in range(nm):
            for q in range(nm - p):
                for r in range(nm - p - q):
                    t = [(_mod_a(p, a), _mod_b(p, q, b), _mod_b(p + q, r, c))]
                    if (p, q, r) == (0, 0, 1):
                        t = [(one, one, half_p(c))]
                    elif p == 0 and q == 1:
                        t.append((half_p(a), half_p(b), t[0][2]))
                    terms.append(t)
    V = np.zeros((a.size, len(terms)))
    G = np.zeros((3, a.size, len(terms)))
    for m, ts in enumerate(terms):
        V[:, m] = sum(x[0] * y[0] * t[0] for x, y, t in ts)
        da = sum(x[1] * y[0] * t[0] for x, y, t in ts)
        db = sum(x[0] * y[1] * t[0] for x, y, t in ts)
        dc = sum(x[0] * y[0] * t[1] for x, y, t in ts)
        if shape == "Hex":
            G[:, :, m] = da, db, dc
        elif shape == "Prism":
            G[:, :, m] = 2 * da / (1 - c), db, da * (1 + a) / (1 - c) + dc
        else:
            d0 = 4 * da / ((1 - b) * (1 - c))
            db = 2 * db / (1 - c)
            G[:, :, m] = d0, 0.5 * (1 + a) * d0 + db, 0.5 * (1 + a) * d0 + 0.5 * (1 + b) * db + dc
    return V, G, W


def _chunks(E):
    return [(lo, min(E, lo + 2048)) for lo in range(0, E, 2048)]


def _exact_apply(shape, nm, nq, E, curved, jac, df, lam, x, vel=None, explicit=False):
    dev = x.device
    V, G, W = (torch.from_numpy(t).to(dev) for t in _dense(shape, nm, nq))
    pts = W.numel()
    X = x.double().reshape(E, -1)
    J = torch.from_numpy(jac).reshape(E, -1)
    F = torch.from_numpy(df).reshape(E, -1, 3, 3)  # [element, point, j, d]: dxi_d / dx_j
    out = [[] for _ in range(6 if explicit else 1)]
    for lo, hi in _chunks(E):
        xs, js, fs = X[lo:hi], J[lo:hi].to(dev), F[lo:hi].to(dev)
        wj = W[None] * js
        u = xs @ V.T
        ref = [xs @ G[d].T for d in range(3)]
        grad = [sum(fs[:, :, j, d] * ref[d] for d in range(3)) for j in range(3)]
        weak = sum((wj * sum(fs[:, :, j, d] * grad[j] for j in range(3))) @ G[d] for d in range(3))
        if explicit:
            for o, t in zip(out, [u, *grad, weak, (wj * u) @ V]):
                o.append(t.reshape(-1))
            continue
        v = u
        if vel is not None:
            vs = torch.from_numpy(vel).reshape(E, pts, 3)[lo:hi].to(dev)
            v = u + sum(vs[:, :, j] * grad[j] for j in range(3))
        out[0].append((lam * ((wj * v) @ V) + weak).reshape(-1))
    out = [torch.cat(o) for o in out]
    return out if explicit else out[0]


def exact(case, seed):
    nm, nq, E, shape, single = case["nm"], case["nq"], case["E"], case["shape"], case["single"]
    if case["kind"] == "solve":
        return None
    if case["kind"] == "batch":
        outs = []
        for i, (sh, m, e) in enumerate(_batch_items(case)):
            jac, df = _geometry(case, sh, m + 1, e, False, seed + 1000 * i)
            x = _values(e * _ncoeff(sh, m), single, seed + 1000 * i)
            outs.append(_exact_apply(sh, m, m + 1, e, False, jac, df, _lambda(seed + i), x))
        return outs
    jac, df = _geometry(case, shape, nq, E, case["curved"], seed)
    x = _values(E * _ncoeff(shape, nm), single, seed)
    vel = _velocity(case, seed) if case["kind"] == "advection" else None
    return _exact_apply(shape, nm, nq, E, case["curved"], jac, df, _lambda(seed), x, vel,
                        case["kind"] == "explicit")
