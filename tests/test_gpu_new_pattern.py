"""Matrices with other patterns on a system that keeps data derived from the
pattern of the one before: every solve answers for the matrix that is set."""

import gc

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

N = 150  # 22801 nodes: the arrays of the pattern come from released memory of exactly their sizes


def renumbered(A, parts, seed):
    """The disjoint union of the meshes, the nodes of each numbered anew: the same counts, another pattern."""
    rng = np.random.default_rng(seed)
    out = []
    for X, C in parts:
        order = rng.permutation(X.shape[0]).astype(np.int32)
        Y = np.empty_like(X)
        Y[order] = X
        out.append((Y, np.where(C >= 0, order[np.maximum(C, 0)], -1).astype(np.int32)))
    return A.union_mesh(out)


def new_matrix(A, s, mesh, C, lam):
    bsr = A.BSRFormat(mesh, 1, use_csr=True)
    bsr.compute_sparsity()
    bsr.assemble_heat(A.DeviceArray.from_numpy(np.full(C.shape[0], lam)), 0.1)
    s.set_bsr(bsr)
    row, col, val, _ = bsr.download()
    return bsr, sp.csr_matrix((val, col, row), shape=(s.nb_dof,) * 2)


def residual(M, s, b):
    return np.linalg.norm(b - M @ s.solution().numpy()) / np.linalg.norm(b)


def check_batch(A, s, offs, bs, M, b, what, **kw):
    res, _ = bs.solve(raise_on_failure=False, rtol=1e-8, **kw)
    r = b - M @ s.solution().numpy()
    for q in range(len(offs) - 1):
        cut = slice(offs[q], offs[q + 1])
        assert res[q].converged and np.linalg.norm(r[cut]) <= 1.01e-8 * np.linalg.norm(b[cut]), (what, q)


@pytest.mark.parametrize("path", ["resident", "streaming", "batch", "chunked"])
def test_released_matrix_and_a_renumbered_one(afem_gpu, path):
    """The second matrix takes the handle's address and the device memory of
    the first, released one."""
    print(f"[case] matrix at a released one's addresses: {path}", flush=True)
    A = afem_gpu
    parts = [A.box_mesh(2, n, 0.2, seed=n) for n in (N, 23)]
    meshes = [renumbered(A, parts, turn) for turn in range(4)]
    handles = [A.Mesh(2, X, C) for X, C, _ in meshes]
    n, offs = meshes[0][0].shape[0], meshes[0][2]
    b = np.random.default_rng(1).normal(size=n)
    s = A.DoFLinearSystem(n)
    s.rhs().upload(b)
    bs = A.BatchSolver(s, offs)
    if path == "chunked":
        bs.set_tiles(1, 1)
    for turn in range(4):
        bsr, M = new_matrix(A, s, handles[turn], meshes[turn][1], 1.0 + turn)
        if path in ("batch", "chunked"):
            check_batch(A, s, offs, bs, M, b, turn)
        else:
            for method in (A.SOLVER_PCG_FP64, A.SOLVER_PCG_MIXED):
                r = s.solve(raise_on_failure=False, method=method, rtol=1e-8, spmv_lanes=0 if path == "resident" else -1)
                assert r.converged and residual(M, s, b) <= 1.01e-8, (turn, method)
        del bsr
        gc.collect()


@pytest.mark.parametrize("kw", [dict(), dict(lanes=1), dict(lanes=8), dict(persistent=1), dict(persistent=2)], ids=str)
def test_views_of_other_patterns(afem_gpu, kw):
    """A view at the same addresses with another pattern, and one at other
    addresses with the pattern's counts; the system closes its row starts into
    arrays of its own, which alternate between two addresses."""
    print(f"[case] batch views {kw}", flush=True)
    A = afem_gpu
    sizes = [700, 300]
    offs = np.concatenate([[0], np.cumsum(sizes)])

    def matrix(offsets, seed):
        rng = np.random.default_rng(seed)
        parts = []
        for n in sizes:
            off = [-rng.uniform(0.5, 1.5, n - o) for o in offsets]
            U = sp.diags(off, offsets, shape=(n, n))
            U = U + U.T
            parts.append(U + sp.diags(0.3 - np.asarray(U.sum(axis=1)).ravel()))
        M = sp.block_diag(parts).tocsr()
        M.sort_indices()
        return M

    def arrays(M):
        return [M.indptr.astype(np.int32)[:-1], M.indices.astype(np.int32), M.data]

    # offsets with the same sum: the same number of entries
    mats = [matrix([1, 30], 0), matrix([11, 20], 1), matrix([7, 24], 2)]
    d = [A.DeviceArray.from_numpy(a) for a in arrays(mats[0])]
    s = A.DoFLinearSystem(offs[-1])
    b = np.random.default_rng(1).normal(size=offs[-1])
    s.rhs().upload(b)
    bs = A.BatchSolver(s, offs)
    if "lanes" in kw:
        bs.set_tiles(kw["lanes"], 1)
        kw = {}

    for turn in range(4):
        M = mats[turn % 3]
        for a, v in zip(d, arrays(M)):
            a.upload(v)
        for _ in range(2 if turn else 1):  # the row starts back at the address of the solve before
            s.set_csr_values(*d)
        check_batch(A, s, offs, bs, M, b, turn, **kw)
    other = [A.DeviceArray.from_numpy(a) for a in arrays(mats[2])]
    for a in d:
        a.zero()  # what the old view left behind is no matrix
    s.set_csr_values(*other)
    s.set_csr_values(*other)
    check_batch(A, s, offs, bs, mats[2], b, "other arrays", **kw)
