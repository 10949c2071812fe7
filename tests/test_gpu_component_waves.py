"""The iteration kernels' two forms of the 3x3-block product (a wave per slice, a
wave per component of one slice): rows of one entry up to several groups of
entries, systems of one block row, around a slice and on both sides of the
default rule's lines, 16- and 32-bit columns, with and without the partials'
extra sum, every engine; scalar matrices beside them.  The residual is
recomputed in numpy; its rounding is far below the tolerance."""
import numpy as np
import pytest
import scipy.sparse as sp

import multiscalefemsolver3d_amd as mfs

pytestmark = pytest.mark.gpu


def spd(ctx, nb, bs, wide, seed):
    """Banded SPD blocks, `wide` block columns to each side in the first rows
    and fewer later, a few rows with their diagonal block only."""
    g = np.random.default_rng(seed)
    I, J, V = [], [], []
    for d in range(1, wide + 1):
        m = (nb - d) if d <= 2 else min(nb - d, 150)
        if m <= 0:
            continue
        i = np.arange(m)
        i = i[(i % 17 != 3) & ((i + d) % 17 != 3)]
        for a in range(bs):
            for b in range(bs):
                v = g.uniform(-1.0, 1.0, len(i))
                I += [bs * i + a, bs * (i + d) + b]
                J += [bs * (i + d) + b, bs * i + a]
                V += [v, v]
    n = nb * bs
    A = sp.csr_matrix((np.concatenate(V), (np.concatenate(I), np.concatenate(J))), (n, n)) if V else sp.csr_matrix((n, n))
    A = (A + sp.diags(np.asarray(abs(A).sum(1)).ravel() * 1.1 + 1.0)).tocsr()
    A.sort_indices()
    if bs == 1:
        return mfs.Mat.csr(ctx, A.indptr, A.indices, A.data), A
    blk = A.tobsr((bs, bs))
    blk.sort_indices()
    return mfs.Mat.bsr3(ctx, blk.indptr, blk.indices, blk.data), A


LINE, LINE64 = 400 * 64, 2100 * 64  # block rows at the lines of the default rule, FP32 and FP64


@pytest.mark.parametrize("bs,nb,wide", [(1, 1, 0), (1, 64, 30), (1, 65, 9), (1, 1000, 40),(3, 1, 0), (3, 63, 14), (3, 300, 30), (3, LINE, 2), (3, LINE + 1, 2), (3, LINE64 + 1, 2)])
@pytest.mark.parametrize("env", [{}, {"MFS_COMPONENT_WAVES": "1"}, {"MFS_COMPONENT_WAVES": "0"},
                                 {"MFS_COMPONENT_WAVES": "1", "MFS_NO_COL16": "1", "MFS_FINISH_SUMS": "1"}])
@pytest.mark.parametrize("precision", [mfs.PREC_F64, mfs.PREC_MIXED])
def test_component_products_solve(ctx, monkeypatch, bs, nb, wide, env, precision):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    M, A = spd(ctx, nb, bs, wide, 5)
    n = A.shape[0]
    rhs = np.random.default_rng(6).normal(size=(7, n))
    B = [mfs.Vec(ctx, n, mfs.F64, b) for b in rhs]
    X = [mfs.Vec(ctx, n, mfs.F64) for _ in rhs]
    for method in (mfs.PCG_JACOBI, mfs.MINRES):
        X[0].fill(0.0)
        rep = mfs.Solver(M, method=method, precision=precision, tol=1e-9, maxit=2000).run(B[0], X[0])
        r = rhs[0] - A @ X[0].download()
        assert rep.status == 0 and np.linalg.norm(r) <= 1.01e-9 * np.linalg.norm(rhs[0])
    for k in (1, 2, 4, 7):
        for x in X:
            x.fill(0.0)
        mfs.solve_multi(M, B[:k], X[:k], method=mfs.PCG_JACOBI, precision=precision, tol=1e-9, maxit=2000)
        for b, x in zip(rhs[:k], X[:k]):
            assert np.linalg.norm(b - A @ x.download()) <= 1.01e-9 * np.linalg.norm(b)


def test_fp64_scalar_products_of_six_systems_keep_their_operands_cached(ctx):
    """Six systems of the 64^3 scalar mesh: with one wave per SIMD too many the
    FP64 iteration took 1.86 times the FP32 one (106 and 57 us), against 1.45
    to 1.5 otherwise; the operands and values are twice as wide, the columns
    are the same."""
    n = 64
    xyz, tets = mfs.mesh_box(n)
    bottom = np.arange((n + 1) ** 2, dtype=np.int32)
    S = mfs.Assembly(ctx, mfs.PROBLEM_SCALAR, xyz, tets, fixed_nodes=bottom, fixed_values=np.zeros(len(bottom)))
    S.run(np.exp(0.5 * np.random.default_rng(3).standard_normal(len(tets))))
    B = [mfs.Vec(ctx, S.A.n, mfs.F64, np.random.default_rng(k).standard_normal(S.A.n)) for k in range(6)]
    X = [mfs.Vec(ctx, S.A.n) for _ in B]
    t = []
    for p in (mfs.PREC_F64, mfs.PREC_MIXED):
        best = 1.0
        for _ in range(4):
            for x in X:
                x.fill(0.0)
            reps = mfs.solve_multi(S.A, B, X, check=False, precision=p, tol=1e-30, inner_tol=1e-30, maxit=200)
            best = min(best, max(r.seconds for r in reps) / max(r.iterations for r in reps))
        t.append(best)
    S.close()
    assert t[0] <= 1.65 * t[1], t
