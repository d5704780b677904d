"""The matrix pattern around a hub node: rows that the count pass keeps (up to
32 columns), rows it does not (33 to 49), and hubs of more cells than its
sorting network takes; filled twice, as recomputed sparsity."""

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu


def fan(k, extra):
    """A closed fan of k triangles around node `extra`, numbered between rim
    nodes, with one triangle apart from it."""
    t = 2 * np.pi * np.arange(k) / k
    X = np.zeros((k + 4, 3))
    ids = np.array([i for i in range(k + 1) if i != extra])
    X[ids, 0], X[ids, 1] = np.cos(t), np.sin(t)
    X[k + 1:, :2] = [[3, 0], [4, 0], [3, 1]]
    C = [[extra, ids[i], ids[(i + 1) % k], -1] for i in range(k)] + [[k + 1, k + 2, k + 3, -1]]
    return X, np.array(C, np.int32)


# cells around the hub: its row has one column more
@pytest.mark.parametrize("k", [3, 30, 31, 32, 33, 48, 49, 64, 140])
def test_hub_rows(afem_gpu, k):
    print(f"[case] hub of {k} cells", flush=True)
    A = afem_gpu
    X, C = fan(k, k // 2)
    n = len(X)
    m = A.Mesh(2, X, C)
    b = A.BSRFormat(m, 1, use_csr=True)
    rows = np.repeat(C[:, :3], 3, axis=1).ravel()
    cols = np.tile(C[:, :3], (1, 3)).ravel()
    want = sp.csr_matrix((np.ones(len(rows)), (rows, cols)), shape=(n, n))
    want.sort_indices()
    for _ in range(2):
        b.compute_sparsity()
        row, col, _, nzr = b.download()
        assert np.array_equal(row, want.indptr)
        assert np.array_equal(col, want.indices)
        assert np.array_equal(nzr, np.diff(want.indptr))
    s = A.DoFLinearSystem(n)
    b.assemble_laplace(None, 1.0, s.rhs())
    _, _, val, _ = b.download()
    K = sp.csr_matrix((val, want.indices, want.indptr), shape=(n, n))
    # constants are in the kernel, and a hub's entry is the sum of its rim entries (2 rounded terms each)
    assert np.abs(K @ np.ones(n)).max() <= 4 * k * np.finfo(float).eps * np.abs(val).max()
