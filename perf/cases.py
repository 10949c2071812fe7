"""Workloads that stand for what users of this library have it do.

Every case is one call chain through the public Python binding.  The sizes
come from the library's own benchmark, tests and configurations; `draw` gives
more cases of the same ranges.

  poisson   scalar Laplace with inclusions (the ElectroStatic driver's system):
            Jacobi-PCG from the Dirichlet start vector.
  elastic   one load step of a Mechanical driver: new moduli are assembled,
            the system is solved, the displacement is read back.
  minres    the reference element convention's operator with MINRES, the
            solver the drop-in routes the driver's solves to.
  loads     the homogenisation driver's load cases, one matrix, k right-hand
            sides.
  nonsym    upwind convection-diffusion with BiCGStab or restarted GMRES.
  operator  assembly at memory-bound size and the bare operator (power
            iteration: SpMV, dot, axpby).
  msfem     the offline stage of the multiscale method: cell assembly, the 24
            local problems of every cell, the coarse element matrices.
  pipeline  a whole small MsFEM run: offline stage, coarse system, coarse
            solve, fine displacement of every cell.
  learned   the batched solve from the network's initial guess: features,
            inference, guess, mixed solve, coarse matrices.
  train     one epoch of the network's training on device-resident samples.
"""
import math

import numpy as np
import torch

import multiscalefemsolver3d_amd as mfs
from multiscalefemsolver3d_amd import learned

NU = 0.3
_CTX = None


def _ctx():
    """One context per process, as a user's program keeps it."""
    global _CTX
    if _CTX is None:
        _CTX = mfs.Context(0)
    return _CTX


def listed():
    return [
        # the smallest solve of the tests: launches and host round trips
        dict(name="poisson12 f64", kind="poisson", n=12, precision="f64", tol=1e-10),
        # the benchmark's Laplace system, FP32 iterations in FP64 refinement
        dict(name="poisson64 mixed", kind="poisson", n=64, precision="mixed", tol=1e-10),
        # a Mechanical load step: upload of the moduli, assembly, FP64 PCG
        dict(name="elastic40 f64", kind="elastic", n=40, precision="f64", tol=1e-11),
        # the 20^3 configuration's operator in the reference's convention
        dict(name="minres20 mixed", kind="minres", n=20, precision="mixed", tol=1e-10),
        # six load cases of the homogenisation driver
        dict(name="loads24 mixed", kind="loads", n=24, k=6, precision="mixed", tol=1e-10),
        # non-symmetric system of the benchmark
        dict(name="nonsym512 bicgstab", kind="nonsym", m=512, method="bicgstab", precision="f64", peclet=200.0,
             tol=1e-9),
        # assembly and FP32 products of an operator larger than the caches
        dict(name="operator80 f32", kind="operator", n=80, precision="f32", steps=10),
        # the 16^3-cell configuration, n ~ U{6..10}, Q1 traces
        dict(name="msfem16 mixed", kind="msfem", nc=16, n_lo=6, n_hi=10, precision="mixed", trace="q1", tol=1e-8),
        # the plain FP64 batch the benchmark compares with, cells of 8^3
        dict(name="msfem8 f64", kind="msfem", nc=8, n_lo=8, n_hi=8, precision="f64", trace="q1", tol=1e-8),
        # reference edge -> face -> volume traces
        dict(name="msfem10 traces", kind="msfem", nc=10, n_lo=4, n_hi=9, precision="mixed", trace="reference",
             tol=1e-8),
        # a whole small multiscale run with its coarse solve and downscaling
        dict(name="pipeline3", kind="pipeline", nc=3, n=5, precision="mixed", tol=1e-11),
        # the learned-guess step of the benchmark on 4,096 cells of 8^3
        dict(name="learned4096", kind="learned", cells=4096, n=8, hidden=256, layers=4, tol=1e-8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["poisson", "poisson", "elastic", "minres", "loads", "nonsym", "operator", "msfem", "msfem",
                       "msfem", "pipeline", "learned", "train"])
    prec = rng.choice(["f64", "mixed"])
    if kind == "poisson":
        return dict(kind=kind, n=_log_int(rng, 6, 64), precision=prec, tol=1e-10)
    if kind == "elastic":
        return dict(kind=kind, n=_log_int(rng, 5, 40), precision=prec, tol=1e-11)
    if kind == "minres":
        return dict(kind=kind, n=_log_int(rng, 5, 20), precision=prec, tol=1e-10)
    if kind == "loads":
        return dict(kind=kind, n=_log_int(rng, 6, 26), k=rng.randint(2, 8), precision=prec, tol=1e-10)
    if kind == "nonsym":
        return dict(kind=kind, m=_log_int(rng, 40, 512), method=rng.choice(["bicgstab", "gmres"]), precision=prec,
                    peclet=float(rng.choice([20.0, 80.0, 200.0])), tol=1e-9)
    if kind == "operator":
        return dict(kind=kind, n=_log_int(rng, 10, 80), precision=rng.choice(["f32", "f64"]), steps=rng.randint(5, 10))
    if kind == "msfem":
        lo = rng.randint(3, 9)
        return dict(kind=kind, nc=_log_int(rng, 2, 12), n_lo=lo, n_hi=min(10, lo + rng.randint(0, 4)), precision=prec,
                    trace=rng.choice(["q1", "q1", "reference"]), tol=1e-8)
    if kind == "pipeline":
        return dict(kind=kind, nc=rng.randint(2, 4), n=rng.randint(3, 6), precision=prec, tol=1e-11)
    if kind == "learned":
        return dict(kind=kind, cells=_log_int(rng, 200, 4096), n=rng.randint(4, 8), hidden=rng.choice([128, 256]),
                    layers=rng.randint(3, 4), tol=1e-8)
    return dict(kind="train", samples=_log_int(rng, 512, 4096), n=rng.randint(4, 8), hidden=rng.choice([128, 256]),
                layers=rng.randint(3, 4), batch=rng.choice([128, 256]))


# ---------------------------------------------------------------------------
# Inputs (seeded, numpy / torch only, shared by prepare and exact)
# ---------------------------------------------------------------------------
PERM = ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0))


def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _inclusions(n, seed):
    """Conductivity per tet: 1 with 200 spherical inclusions of 100."""
    g = np.random.default_rng([seed, 1])
    ctr = torch.tensor(g.uniform(0, 1, (200, 3)), device=_dev())
    rad = torch.tensor(g.uniform(0.02, 0.06, 200), device=_dev())
    hexes = torch.arange(n ** 3, device=_dev())
    base = torch.stack([hexes % n, (hexes // n) % n, hexes // (n * n)], 1).double()
    sig = torch.ones(n ** 3, 6, dtype=torch.float64, device=_dev())
    for p, perm in enumerate(PERM):
        off = torch.zeros(3, dtype=torch.float64)
        for v in range(3):  # centroid: axis stepped v-th is held by 3 - v of the 4 vertices
            off[perm[v]] = (3 - v) / 4.0
        c = (base + off.to(_dev())) / n
        hit = torch.zeros(n ** 3, dtype=torch.bool, device=_dev())
        for q in range(200):
            hit |= ((c - ctr[q]) ** 2).sum(1) < rad[q] ** 2
        sig[:, p] = torch.where(hit, 100.0, 1.0)
    return sig.reshape(-1).cpu().numpy()


def _moduli(count, seed, sigma=0.5):
    """Lognormal Young's modulus per tet around 1 GPa."""
    return np.exp(math.log(1e9) + sigma * np.random.default_rng([seed, 2]).standard_normal(count))


def _bottom(n):
    return np.arange((n + 1) ** 2, dtype=np.int32)


def _top(n):
    return _bottom(n) + np.int32((n + 1) ** 2 * n)


def _top_load(n, pressure):
    """Nodal forces of a uniform pressure on the top face."""
    f = np.zeros(((n + 1) ** 3, 3))
    s = n + 1
    for i0, j0 in ((0, 0), (1, 0), (1, 1), (0, 0), (0, 1), (1, 1)):  # the two triangles of each square
        i, j = np.meshgrid(np.arange(n) + i0, np.arange(n) + j0, indexing="ij")
        np.add.at(f[:, 2], (i + s * (j + s * n)).ravel(), -pressure * 0.5 / n ** 2 / 3.0)
    return f


def _load_cases(n, k, seed):
    """k nodal load fields: a smooth random field per component, none on the clamped face."""
    g = np.random.default_rng([seed, 3])
    t = np.arange(n + 1) / n
    Z, Y, X = np.meshgrid(t, t, t, indexing="ij")
    out = []
    for _ in range(k):
        f = np.empty(((n + 1) ** 3, 3))
        for a in range(3):
            w = g.normal(size=4)
            ph = g.uniform(0, 2 * math.pi, 3)
            f[:, a] = (w[0] + w[1] * np.cos(3 * X + ph[0]) + w[2] * np.cos(4 * Y + ph[1]) +
                       w[3] * np.cos(5 * Z + ph[2])).ravel() * 1e6 / n ** 3
        f[_bottom(n)] = 0.0
        out.append(f)
    return out


def _cell_sizes(case, seed):
    return np.random.default_rng([seed, 4]).integers(case["n_lo"], case["n_hi"] + 1, case["nc"] ** 3).astype(np.int32)


def _cell_grid(nc):
    i = np.arange(nc ** 3)
    return np.stack([i % nc, (i // nc) % nc, i // (nc * nc)], 1) / nc


def _convection(m, peclet):
    """Five upwind 5-point coefficients (diagonal, x-, x+, y-, y+) on an m x m grid."""
    h = 1.0 / (m + 1)
    cx, cy = peclet, 0.5 * peclet
    return 4.0 / h ** 2 + (cx + cy) / h, -1 / h ** 2 - cx / h, -1 / h ** 2, -1 / h ** 2 - cy / h, -1 / h ** 2


def _convection_csr(m, peclet):
    d, xm, xp, ym, yp = _convection(m, peclet)
    r = np.arange(m * m)
    i, j = r % m, r // m
    cols = np.stack([r - m, r - 1, r, r + 1, r + m], 1)
    ok = np.stack([j > 0, i > 0, np.ones_like(i, bool), i < m - 1, j < m - 1], 1)
    vals = np.broadcast_to(np.array([ym, xm, d, xp, yp]), cols.shape)
    rowptr = np.concatenate([[0], np.cumsum(ok.sum(1))]).astype(np.int32)
    return rowptr, cols[ok].astype(np.int32), np.ascontiguousarray(vals[ok])


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
_METHOD = {"bicgstab": mfs.BICGSTAB, "gmres": mfs.GMRES}
_PREC = {"f64": mfs.PREC_F64, "mixed": mfs.PREC_MIXED}


def _elastic_assembly(n, convention, loaded=True):
    xyz, tets = mfs.mesh_box(n)
    tris = mfs.box_face_tris(n, n, n, 5) if loaded else None
    return mfs.Assembly(_ctx(), mfs.PROBLEM_ELASTIC, xyz, tets, renumber=True, convention=convention,
                        fixed_nodes=_bottom(n), fixed_values=np.zeros((len(_bottom(n)), 3)), tris=tris,
                        traction=np.tile([0.0, 0.0, -1e6], (len(tris), 1)) if loaded else None)


def prepare(case, seed):
    kind, ctx = case["kind"], _ctx()
    st = dict(case=case)
    prec = _PREC.get(case.get("precision"))
    if kind == "poisson":
        n = case["n"]
        xyz, tets = mfs.mesh_box(n)
        vals = np.concatenate([np.zeros((n + 1) ** 2), np.ones((n + 1) ** 2)])
        S = mfs.Assembly(ctx, mfs.PROBLEM_SCALAR, xyz, tets, fixed_nodes=np.concatenate([_bottom(n), _top(n)]),
                         fixed_values=vals)
        S.run(_inclusions(n, seed))
        st.update(S=S, x=mfs.Vec(ctx, S.A.n), solver=mfs.Solver(S.A, precision=prec, tol=case["tol"]))
    elif kind in ("elastic", "minres"):
        n = case["n"]
        textbook = kind == "elastic"
        S = _elastic_assembly(n, mfs.ELEM_TEXTBOOK if textbook else mfs.ELEM_REFERENCE)
        if textbook:
            E = _moduli(6 * n ** 3, seed)
        else:
            E = np.full(6 * n ** 3, 1e9 * (1.0 + 0.5 * np.random.default_rng([seed, 5]).uniform()))
        S.run(E, NU)
        st.update(S=S, E=E, map=S.node_map(), x=mfs.Vec(ctx, S.A.n),
                  solver=mfs.Solver(S.A, method=mfs.PCG_JACOBI if textbook else mfs.MINRES, precision=prec,
                                    tol=case["tol"]))
    elif kind == "loads":
        n, k = case["n"], case["k"]
        S = _elastic_assembly(n, mfs.ELEM_TEXTBOOK, loaded=False)
        S.run(_moduli(6 * n ** 3, seed), NU)
        m = S.node_map()
        b = []
        for f in _load_cases(n, k, seed):
            g = np.empty_like(f)
            g[m] = f
            b.append(mfs.Vec(ctx, S.A.n, mfs.F64, g))
        st.update(S=S, map=m, b=b, x=[mfs.Vec(ctx, S.A.n) for _ in b],
                  desc=mfs.solve_desc(precision=prec, tol=case["tol"]))
    elif kind == "nonsym":
        rowptr, col, val = _convection_csr(case["m"], case["peclet"])
        A = mfs.Mat.csr(ctx, rowptr, col, val)
        b = mfs.Vec(ctx, A.n, mfs.F64, np.random.default_rng([seed, 6]).standard_normal(A.n))
        st.update(A=A, b=b, x=mfs.Vec(ctx, A.n),
                  solver=mfs.Solver(A, method=_METHOD[case["method"]], precision=prec, tol=case["tol"]))
    elif kind == "operator":
        n = case["n"]
        p = mfs.F32 if case["precision"] == "f32" else mfs.F64
        S = _elastic_assembly(n, mfs.ELEM_TEXTBOOK)
        g = np.random.default_rng([seed, 7]).standard_normal(3 * (n + 1) ** 3)
        m = S.node_map()
        x0 = np.empty((len(m), 3))
        x0[m] = g.reshape(-1, 3)
        st.update(S=S, E=_moduli(6 * n ** 3, seed), prec=p, map=m, x0=mfs.Vec(ctx, S.A.n, p, x0),
                  x=mfs.Vec(ctx, S.A.n, p), y=mfs.Vec(ctx, S.A.n, p))
    elif kind == "msfem":
        cn = _cell_sizes(case, seed)
        nt = int((6 * cn.astype(np.int64) ** 3).sum())
        trace = mfs.TRACE_REFERENCE if case["trace"] == "reference" else mfs.TRACE_Q1
        st.update(B=mfs.Batch(ctx, cn, _cell_grid(case["nc"]), 1.0 / case["nc"], _moduli(nt, seed, 1.0), NU,
                              trace=trace), prec=prec)
    elif kind == "pipeline":
        nc, n = case["nc"], case["n"]
        st.update(B=mfs.Batch(ctx, np.full(nc ** 3, n, np.int32), _cell_grid(nc), 1.0 / nc,
                              _moduli(6 * n ** 3 * nc ** 3, seed), NU, convention=mfs.ELEM_TEXTBOOK),
                  prec=prec, nn=(nc + 1) ** 3)
    elif kind in ("learned", "train"):
        n = case["n"]
        count = case["cells"] if kind == "learned" else case["samples"]
        nt, nout = 6 * n ** 3, 72 * (n - 1) ** 3
        E = _moduli(count * nt, seed, 1.0)
        origin = np.zeros((count, 3))
        origin[:, 0] = np.arange(count) / 32
        B = mfs.Batch(ctx, np.full(count, n, np.int32), origin, 1.0 / 32, E)
        B.assemble()
        net = mfs.MLP(ctx, [nt] + [case["hidden"]] * (case["layers"] - 1) + [nout], seed=11)
        # training pairs: for `train` the cells themselves, for `learned` the first 256 cells
        few = count if kind == "train" else min(count, 256)
        Bt = B if kind == "train" else mfs.Batch(ctx, np.full(few, n, np.int32), origin[:few], 1.0 / 32, E[:few * nt])
        if Bt is not B:
            Bt.assemble()
        Bt.solve(precision=mfs.PREC_MIXED, tol=1e-8)
        X, T = mfs.Vec(ctx, few * nt, mfs.F32), mfs.Vec(ctx, few * nout, mfs.F32)
        Bt.features(X, learned.MU_LOGE, learned.SIGMA_LOGE)
        Bt.targets(T)
        Bt.close()
        if kind == "train":
            st.update(net=net, X=X, T=T, init=net.get_params())
        else:
            net.train_vec(few, X, T, min(few, 64), 20, seed=3)
            model = learned.Trained(net, n, {mfs.PREC_MIXED: {}, mfs.PREC_F64: {}}, {})
            st.update(B=B, L=learned.LearnedSolver(ctx, model, B, count, case["tol"]), net=net)
    return st


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "poisson":
        st["x"].copy_from(st["S"].x0)
        st["solver"].run(st["S"].b, st["x"])
        return st["x"].download()
    if kind in ("elastic", "minres"):
        st["S"].run(st["E"], NU)
        st["x"].copy_from(st["S"].x0)
        st["solver"].run(st["S"].b, st["x"])
        return st["x"].download().reshape(-1, 3)[st["map"]]
    if kind == "loads":
        import ctypes
        k = case["k"]
        for x in st["x"]:
            x.fill(0.0)
        reps = (mfs.SolveReport * k)()
        bs, xs = (ctypes.c_void_p * k)(*[b.h for b in st["b"]]), (ctypes.c_void_p * k)(*[x.h for x in st["x"]])
        if mfs.lib.mfs_solve_multi(st["S"].A.h, ctypes.byref(st["desc"]), k, bs, xs, reps) != 0:
            raise RuntimeError(mfs.lib.mfs_last_error())
        return [x.download().reshape(-1, 3)[st["map"]] for x in st["x"]]
    if kind == "nonsym":
        st["x"].fill(0.0)
        st["solver"].run(st["b"], st["x"])
        return st["x"].download()
    if kind == "operator":
        S, x, y = st["S"], st["x"], st["y"]
        S.run(st["E"], NU)
        x.copy_from(st["x0"])
        rayleigh = 0.0
        for _ in range(case["steps"]):
            nx = math.sqrt(mfs.dot(x, x))
            S.A.spmv(x, y, st["prec"])
            rayleigh = mfs.dot(x, y) / nx ** 2
            mfs.axpby(1.0 / nx / abs(rayleigh), y, 0.0, x)
        out = x.download().reshape(-1, 3)[st["map"]]
        return (out.astype(np.float32), np.float32(rayleigh)) if st["prec"] == mfs.F32 else (out, rayleigh)
    if kind == "msfem":
        B = st["B"]
        B.assemble()
        B.solve(precision=st["prec"], tol=case["tol"], check=False)
        return B.coarse_matrices()
    if kind == "pipeline":
        B = st["B"]
        B.assemble()
        B.solve(precision=st["prec"], tol=case["tol"], check=False)
        load = B.top_traction([0.0, 0.0, -1e6], st["nn"])
        nf = (case["nc"] + 1) ** 2
        A, b, x = B.coarse_system(B.coarse_matrices(), load, np.arange(nf, dtype=np.int32), np.zeros((nf, 3)))
        mfs.Solver(A, tol=1e-12).run(b, x)
        u = x.download()
        return [u] + [np.stack([B.downscale(u, c) for c in range(B.ncells)])]
    if kind == "learned":
        st["L"].solve()
        return st["B"].coarse_matrices()
    net = st["net"]
    net.set_params(st["init"])
    loss = net.train_vec(case["samples"], st["X"], st["T"], case["batch"], 1, seed=3)
    return [np.float32(loss)] + [a for W, b in net.get_params() for a in (W, b)]


# ---------------------------------------------------------------------------
# work: inputs read once, outputs written once; the arithmetic of one product
# with the operator (an iterative solve needs at least one per right-hand side)
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind in ("poisson", "elastic", "minres", "loads", "operator"):
        n = case["n"]
        bs = 1 if kind == "poisson" else 3
        nnzb = 15 * n ** 3 + 29 * n * n + 17 * n + 1  # nodes + 2 edges of the Freudenthal mesh
        dof = bs * (n + 1) ** 3
        k = case.get("k", case.get("steps", 1))
        sv = 4 if case["precision"] == "f32" else 8
        by = nnzb * bs * bs * sv * (k if kind == "operator" else 1) + 2 * dof * 8 * k
        if kind in ("elastic", "minres", "operator"):
            by += 8 * 6 * n ** 3
        return dict(bytes=by, flops=2 * nnzb * bs * bs * k)
    if kind == "nonsym":
        return dict(bytes=(5 * 12 + 16) * case["m"] ** 2, flops=2 * 10 * case["m"] ** 2)
    if kind in ("msfem", "pipeline", "learned"):
        if kind == "msfem":
            cells, n = case["nc"] ** 3, 0.5 * (case["n_lo"] + case["n_hi"])
        else:
            cells, n = (case["nc"] ** 3 if kind == "pipeline" else case["cells"]), case["n"]
        nodes = (n - 1) ** 3
        # moduli in, bases in FP64 and coarse matrices out; one stencil product per
        # problem and the Galerkin product of 24 functions
        flops = cells * (24 * nodes * 270 + 6 * n ** 3 * 9 * 24 * 24 * 2)
        if kind == "learned":
            d = [6 * n ** 3] + [case["hidden"]] * (case["layers"] - 1) + [72 * nodes]
            flops += 2 * cells * sum(a * b for a, b in zip(d, d[1:]))
        return dict(bytes=cells * (6 * n ** 3 * 8 + nodes * 72 * 8 + 576 * 8), flops=flops)
    d = [6 * case["n"] ** 3] + [case["hidden"]] * (case["layers"] - 1) + [72 * (case["n"] - 1) ** 3]
    w = sum(a * b for a, b in zip(d, d[1:]))
    s = case["samples"] // case["batch"] * case["batch"]
    return dict(bytes=4 * s * (d[0] + d[-1]) + s // case["batch"] * 24 * w, flops=6 * s * w)


# ---------------------------------------------------------------------------
# exact: the same results in 64 bits, from the mesh and the element formulas
# ---------------------------------------------------------------------------
def _tets(n, s):
    """(4, n^3) node numbers of each of the six tets of a hex, per tet shape."""
    h = torch.arange(n ** 3, device=_dev())
    c = [h % n, (h // n) % n, h // (n * n)]
    out = []
    for perm in PERM:
        at = [t.clone() for t in c]
        nodes = [at[0] + s * (at[1] + s * at[2])]
        for ax in perm:
            at[ax] = at[ax] + 1
            nodes.append(at[0] + s * (at[1] + s * at[2]))
        out.append(torch.stack(nodes))
    return out


class _Operator:
    """Matrix-free P1 operator of the n^3 Freudenthal mesh of a cube of edge `size`.

    The gradient of a P1 function on a tet is the difference along each of its
    three axis-parallel edges."""

    def __init__(self, n, coef, bs, textbook=True, size=1.0):
        self.n, self.bs, self.textbook, self.h = n, bs, textbook, size / n
        self.nodes = _tets(n, n + 1)
        c = torch.tensor(coef, device=_dev(), dtype=torch.float64).reshape(-1, 6)
        v = self.h ** 3 / 6.0
        self.c = [c[:, p] * v for p in range(6)]
        self.lam, self.mu = NU / ((1 + NU) * (1 - 2 * NU)), 0.5 / (1 + NU)

    def __call__(self, u):
        y = torch.zeros_like(u)
        for p, perm in enumerate(PERM):
            un = u[self.nodes[p]]  # (4, hexes, bs)
            g = [None] * 3
            for v, ax in enumerate(perm):
                g[ax] = (un[v + 1] - un[v]) / self.h
            c = self.c[p][:, None]
            if self.bs == 1:
                f = [c * g[b] for b in range(3)]
            else:
                G = torch.stack(g, 2)  # G[:, a, b] = d_b u_a
                tr = (G[:, 0, 0] + G[:, 1, 1] + G[:, 2, 2])[:, None, None] * torch.eye(3, device=u.device,
                                                                                      dtype=u.dtype)
                Gt = G.transpose(1, 2)
                s = self.lam * tr + self.mu * (G + Gt) if self.textbook else self.lam * Gt + self.mu * (G + tr)
                s = s * c[:, :, None]
                f = [s[:, :, b] for b in range(3)]
            for v, ax in enumerate(perm):
                y.index_add_(0, self.nodes[p][v + 1], f[ax] / self.h)
                y.index_add_(0, self.nodes[p][v], -f[ax] / self.h)
        return y


def _cg(A, b, diag, tol=1e-14, rounds=6, cap=20000):
    """Jacobi-PCG with residual replacement, per trailing column block as one system."""
    x = torch.zeros_like(b)
    bb = b.norm()
    for _ in range(rounds):
        r = b - A(x)
        if r.norm() <= tol * bb:
            break
        z = r / diag
        p, rz = z.clone(), (r * z).sum()
        target = max(1e-9, 0.3 * tol * float(bb) / float(r.norm())) * r.norm()
        for it in range(cap):
            q = A(p)
            al = rz / (p * q).sum()
            x += al * p
            r -= al * q
            if it % 16 == 15 and not bool(r.norm() > target):
                break
            z = r / diag
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
    return x


def _bicgstab(A, b, diag, tol=1e-14, rounds=12, cap=8000):
    x = torch.zeros_like(b)
    bb = b.norm()
    for _ in range(rounds):
        r = b - A(x)
        if r.norm() <= tol * bb:
            break
        target = max(1e-8, 0.3 * tol * float(bb) / float(r.norm())) * r.norm()
        r0, p, rho = r.clone(), r.clone(), (r * r).sum()
        for it in range(cap):
            ph = p / diag
            v = A(ph)
            al = rho / (r0 * v).sum()
            s = r - al * v
            sh = s / diag
            t = A(sh)
            om = (t * s).sum() / (t * t).sum()
            x += al * ph + om * sh
            r = s - om * t
            if it % 16 == 15 and not bool(r.norm() > target):
                break
            new = (r0 * r).sum()
            p = r + (new / rho) * (al / om) * (p - om * v)
            rho = new
    return x


def _diagonal(op, bs):
    """Diagonal by probing the 27-colouring of the mesh's nodes."""
    s = op.n + 1
    v = torch.arange(s ** 3, device=_dev())
    colour = (v % s) % 3 + 3 * (((v // s) % s) % 3) + 9 * ((v // (s * s)) % 3)
    d = torch.zeros(s ** 3, bs, device=_dev(), dtype=torch.float64)
    for a in range(bs):
        for c in range(27):
            e = torch.zeros_like(d)
            e[colour == c, a] = 1.0
            d[:, a] += torch.where(colour == c, op(e)[:, a], 0.0)
    return d


def _solve_fixed(op, bs, fixed, x0, f):
    """Solve with the nodes `fixed` held at x0 and nodal loads f."""
    free = torch.ones(f.shape[0], 1, device=_dev(), dtype=torch.float64)
    free[torch.tensor(fixed, device=_dev(), dtype=torch.long)] = 0.0
    diag = _diagonal(op, bs)
    diag = torch.where(free > 0, diag, torch.ones_like(diag))
    b = free * (f - op(x0))
    return x0 + _cg(lambda u: free * op(free * u) + (1 - free) * u, b, diag)


def _dense_cells(case, seed):
    """Local bases, coarse matrices and top loads of the pipeline's cells, dense."""
    nc, n = case["nc"], case["n"]
    s, m = n + 1, n - 1
    E = _moduli(6 * n ** 3 * nc ** 3, seed).reshape(nc ** 3, -1)
    t = np.arange(s) / n
    Z, Y, X = np.meshgrid(t, t, t, indexing="ij")
    hat = np.stack([((X if c & 1 else 1 - X) * (Y if c & 2 else 1 - Y) * (Z if c & 4 else 1 - Z)).ravel()
                    for c in range(8)], 1)
    g = np.zeros((s ** 3, 3, 24))
    for c in range(8):
        for d in range(3):
            g[:, d, 3 * c + d] = hat[:, c]
    v = np.arange(s ** 3)
    i, j, k = v % s, (v // s) % s, v // (s * s)
    inner = (i > 0) & (i < n) & (j > 0) & (j < n) & (k > 0) & (k < n)
    dof = np.nonzero(np.repeat(inner, 3))[0]
    eye = torch.eye(3 * s ** 3, device=_dev(), dtype=torch.float64)
    bases, Kc = [], []
    for c in range(nc ** 3):
        op = _Operator(n, E[c], 3, True, 1.0 / nc)
        K = torch.stack([op(col.reshape(-1, 3)).reshape(-1) for col in eye], 1).cpu().numpy()
        phi = g.reshape(-1, 24).copy()
        phi[dof] = 0.0
        phi[dof] = np.linalg.solve(K[np.ix_(dof, dof)], -(K @ phi)[dof])
        bases.append(phi)
        Kc.append(phi.T @ K @ phi)
    return bases, Kc, hat


def exact(case, seed):
    kind = case["kind"]
    if kind == "poisson":
        n = case["n"]
        op = _Operator(n, _inclusions(n, seed), 1)
        x0 = torch.zeros((n + 1) ** 3, 1, device=_dev(), dtype=torch.float64)
        x0[torch.tensor(_top(n), device=_dev(), dtype=torch.long)] = 1.0
        fixed = np.concatenate([_bottom(n), _top(n)])
        return _solve_fixed(op, 1, fixed, x0, torch.zeros_like(x0)).reshape(-1).cpu().numpy()
    if kind in ("elastic", "minres"):
        n = case["n"]
        E = _moduli(6 * n ** 3, seed) if kind == "elastic" else np.full(
            6 * n ** 3, 1e9 * (1.0 + 0.5 * np.random.default_rng([seed, 5]).uniform()))
        op = _Operator(n, E, 3, kind == "elastic")
        f = torch.tensor(_top_load(n, 1e6), device=_dev())
        return _solve_fixed(op, 3, _bottom(n), torch.zeros_like(f), f).cpu().numpy()
    if kind == "loads":
        n = case["n"]
        op = _Operator(n, _moduli(6 * n ** 3, seed), 3)
        return [_solve_fixed(op, 3, _bottom(n), torch.zeros((n + 1) ** 3, 3, device=_dev(), dtype=torch.float64),
                             torch.tensor(f, device=_dev())).cpu().numpy() for f in _load_cases(n, case["k"], seed)]
    if kind == "nonsym":
        m = case["m"]
        d, xm, xp, ym, yp = _convection(m, case["peclet"])
        b = torch.tensor(np.random.default_rng([seed, 6]).standard_normal(m * m), device=_dev()).reshape(m, m)

        def A(u):
            y = d * u
            y[:, 1:] += xm * u[:, :-1]
            y[:, :-1] += xp * u[:, 1:]
            y[1:] += ym * u[:-1]
            y[:-1] += yp * u[1:]
            return y

        return _bicgstab(A, b, d).reshape(-1).cpu().numpy()
    if kind == "operator":
        n = case["n"]
        op = _Operator(n, _moduli(6 * n ** 3, seed), 3)
        free = torch.ones((n + 1) ** 3, 1, device=_dev(), dtype=torch.float64)
        free[torch.tensor(_bottom(n), device=_dev(), dtype=torch.long)] = 0.0
        x = torch.tensor(np.random.default_rng([seed, 7]).standard_normal(3 * (n + 1) ** 3), device=_dev()).reshape(-1, 3)
        ray = 0.0
        for _ in range(case["steps"]):
            nx = float(x.norm())
            y = free * op(free * x) + (1 - free) * x
            ray = float((x * y).sum()) / nx ** 2
            x = y / nx / abs(ray)
        return x.cpu().numpy(), ray
    if kind == "pipeline" and case["nc"] ** 3 * (case["n"] + 1) ** 3 <= 8000:
        nc, n = case["nc"], case["n"]
        bases, Kc, hat = _dense_cells(case, seed)
        sc, s = nc + 1, n + 1
        N = sc ** 3
        A, f = np.zeros((3 * N, 3 * N)), np.zeros((N, 3))
        top = _top_load(n, 1e6)[:, 2] / nc ** 2  # nodal forces on a cell's top face
        node = []
        for c in range(nc ** 3):
            I, J, K = c % nc, (c // nc) % nc, c // (nc * nc)
            q = np.array([(I + (b & 1)) + sc * ((J + ((b >> 1) & 1)) + sc * (K + (b >> 2))) for b in range(8)])
            node.append(q)
            d = (3 * q[:, None] + np.arange(3)).ravel()
            A[np.ix_(d, d)] += Kc[c]
            if K == nc - 1:
                f[q, 2] += hat.T @ top
        free = np.arange(3 * sc * sc, 3 * N)  # the bottom plane's nodes come first
        u = np.zeros(3 * N)
        u[free] = np.linalg.solve(A[np.ix_(free, free)], f.ravel()[free])
        fine = [bases[c] @ u.reshape(-1, 3)[node[c]].ravel() for c in range(nc ** 3)]
        return [u, np.stack(fine)]
    return None
