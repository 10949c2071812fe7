"""The two-kernel MINRES step at its edges: block sizes 1 and 3, systems of one
row up to several slices, 16- and 32-bit columns, with and without the
partials' extra sum, graph and direct launches, an iteration cap in and at the
end of a chunk, and a zero right-hand side.  The residual is recomputed in
numpy from the exported matrix; its rounding is far below the tolerance."""
import numpy as np
import pytest
import scipy.sparse as sp

import multiscalefemsolver3d_amd as mfs

pytestmark = pytest.mark.gpu


def indefinite(ctx, nb, bs, seed):
    """Symmetric indefinite banded matrix with a positive diagonal (the
    preconditioner must be SPD): neighbouring blocks coupled in pairs by 2 I
    (eigenvalues near 3 and -1) and weak random couplings further out."""
    g = np.random.default_rng(seed)
    A = sp.lil_matrix((nb * bs, nb * bs))
    for d in (1, 2, 7):
        for i in range(nb - d):
            B = g.normal(size=(bs, bs)) * 0.03
            if d == 1 and i % 2 == 0:
                B += 2.0 * np.eye(bs)
            A[bs * i:bs * i + bs, bs * (i + d):bs * (i + d) + bs] = B
            A[bs * (i + d):bs * (i + d) + bs, bs * i:bs * i + bs] = B.T
    A.setdiag(1.0 + g.uniform(-0.1, 0.1, nb * bs))
    A = A.tocsr()
    if bs == 1:
        A.sort_indices()
        return mfs.Mat.csr(ctx, A.indptr, A.indices, A.data), A
    blk = A.tobsr((bs, bs))
    blk.sort_indices()
    return mfs.Mat.bsr3(ctx, blk.indptr, blk.indices, blk.data), A


@pytest.mark.parametrize("bs,nb", [(1, 1), (1, 64), (1, 1500), (3, 1), (3, 65), (3, 700)])
@pytest.mark.parametrize("env", [{}, {"MFS_NO_GRAPH": "1"}, {"MFS_FINISH_SUMS": "1", "MFS_NO_COL16": "1"}])
@pytest.mark.parametrize("precision", [mfs.PREC_F64, mfs.PREC_MIXED])
def test_minres_solves_indefinite_systems(ctx, monkeypatch, bs, nb, env, precision):
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    M, A = indefinite(ctx, nb, bs, 3)
    b = np.random.default_rng(4).normal(size=A.shape[0])
    B, X = mfs.Vec(ctx, len(b), mfs.F64, b), mfs.Vec(ctx, len(b), mfs.F64)
    S = mfs.Solver(M, method=mfs.MINRES, precision=precision, tol=1e-9, maxit=5000)
    for _ in range(3):  # the graph is replayed from the same start
        X.fill(0.0)
        rep = S.run(B, X)
        r = b - A @ X.download()
        assert rep.status == 0 and np.linalg.norm(r) <= 1.01e-9 * np.linalg.norm(b)
    X.fill(0.0)
    B.fill(0.0)
    assert S.run(B, X).iterations == 0 and not X.download().any()


@pytest.mark.parametrize("cap", [1, 5, 12, 13, 24, 30])
def test_minres_iteration_cap(ctx, cap):
    M, A = indefinite(ctx, 900, 3, 5)
    b = np.random.default_rng(6).normal(size=A.shape[0])
    B, X = mfs.Vec(ctx, len(b), mfs.F64, b), mfs.Vec(ctx, len(b), mfs.F64)
    X.fill(0.0)
    rep = mfs.Solver(M, method=mfs.MINRES, precision=mfs.PREC_F64, tol=1e-14, maxit=cap).run(B, X, check=False)
    assert rep.iterations == cap and rep.status == -3
    r = np.linalg.norm(b - A @ X.download()) / np.linalg.norm(b)
    assert abs(r - rep.true_relres) <= 1e-10 and r < 1.0
