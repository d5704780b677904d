"""Solves whose vectors stay on the chip (one launch per solve) against host
references and against the kernels that keep every vector in memory (a
pinned SpMV format selects those).

Both run the same recurrences, so iteration counts agree up to rounding in
the dot products: within max(3, 5 %).  Residuals are checked on the host
with the stated tolerance (1.01 x for the host's own rounding of b - A x).
"""

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

METHODS = {"fp64": 0, "mixed": 1, "cg": 2}


def device_system(A, M):
    M = M.tocsr()
    M.sort_indices()
    d = [A.DeviceArray.from_numpy(a) for a in (M.indptr.astype(np.int32)[:-1], M.indices.astype(np.int32), M.data)]
    s = A.DoFLinearSystem(M.shape[0])
    s.set_csr_values(*d)
    return s, d


def band(n, offsets, shift=0.05, seed=0):
    """Symmetric diagonally dominant matrix with random couplings at the offsets."""
    rng = np.random.default_rng(seed)
    rows, cols, vals = [], [], []
    for o in offsets:
        if o >= n:
            continue
        v = -rng.uniform(0.5, 1.5, n - o)
        i = np.arange(n - o)
        rows += [i, i + o]
        cols += [i + o, i]
        vals += [v, v]
    if rows:
        M = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))), shape=(n, n))
    else:
        M = sp.csr_matrix((n, n))
    d = -np.asarray(M.sum(axis=1)).ravel() * (1 + shift) + shift
    return (M + sp.diags(d)).tocsr()


def check(A, M, method, rtol, norm=0, max_iter=20000):
    rng = np.random.default_rng(1)
    b = rng.normal(size=M.shape[0])
    out = {}
    for lanes in (0, -1):
        s, keep = device_system(A, M)
        s.rhs().upload(b)
        r = s.solve(method=METHODS[method], rtol=rtol, norm=norm, max_iter=max_iter, spmv_lanes=lanes)
        x = s.solution().numpy()
        assert r.converged
        if norm == 0:
            assert np.linalg.norm(b - M @ x) <= 1.01 * rtol * np.linalg.norm(b), (lanes, r.relres)
            assert r.relres <= rtol
        out[lanes] = (r.iterations, x)
    a, g = out[0][0], out[-1][0]
    assert abs(a - g) <= max(3, 0.05 * g), (a, g)
    return out


# rows around one slice, one workgroup (16 slices), one slice per wave on 256
# CUs (262144 rows), and the first rows that need 2, 5 and 9 slices per wave
SIZES = [1, 2, 63, 64, 65, 1023, 1024, 1025, 4097, 131073, 262144, 262145, 524289, 1310721]


@pytest.mark.parametrize("method", ["fp64", "mixed"])
@pytest.mark.parametrize("n", SIZES)
def test_sizes(afem_gpu, n, method):
    print(f"[case] resident n={n} {method}", flush=True)
    check(afem_gpu, band(n, [1, 2, 70], shift=0.3), method, 1e-9 if method == "fp64" else 1e-8)


# pairs per row from none to more than two chunks, odd counts, and offsets
# that need 32 bits
PATTERNS = {"diagonal": (300, []), "one": (1000, [1]), "three_pairs": (1000, [1, 5, 31]),
            "seven_pairs": (5000, [1, 2, 3, 40, 41, 700, 701]), "nine_pairs": (3000, list(range(1, 10))),
            "twenty_pairs": (3000, list(range(1, 21))), "far": (70001, [1, 33000, 40001])}


@pytest.mark.parametrize("method", ["fp64", "mixed", "cg"])
@pytest.mark.parametrize("name", PATTERNS)
def test_patterns(afem_gpu, name, method):
    n, offsets = PATTERNS[name]
    print(f"[case] resident pattern {name} {method}", flush=True)
    check(afem_gpu, band(n, offsets, shift=0.2), method, 1e-9 if method != "mixed" else 1e-8)


@pytest.mark.parametrize("norm", [1, 2])
def test_norms(afem_gpu, norm):
    print(f"[case] resident norm {norm}", flush=True)
    M = band(20000, [1, 2, 150], shift=0.01)
    out = check(afem_gpu, M, "fp64", 1e-10, norm=norm)
    x, y = out[0][1], out[-1][1]
    assert np.linalg.norm(x - y) <= 1e-7 * np.linalg.norm(y)


def test_one_long_row_takes_the_general_kernels(afem_gpu):
    """A dense row would pad its slice's pairs 3000 times over."""
    print("[case] resident long row", flush=True)
    n = 6000
    M = band(n, [1], shift=0.5).tolil()
    M[0, :] = -1e-3
    M[:, 0] = -1e-3
    M[0, 0] = 50.0
    check(afem_gpu, M.tocsr(), "fp64", 1e-10)


def test_more_iterations_than_one_launch(afem_gpu):
    """8192 iterations end a launch: the vectors are kept and the next one goes
    on.  The 1D Laplacian needs about n / 2 iterations; x reaches n^2 / 8 =
    5e7, so b - A x carries up to eps * 4 * 5e7 = 4e-8 of rounding against
    b = 1: the tolerance is 1e-6."""
    print("[case] resident relaunch", flush=True)
    A = afem_gpu
    n = 20000
    M = sp.diags([np.full(n, 2.0), -np.ones(n - 1), -np.ones(n - 1)], [0, 1, -1]).tocsr()
    s, keep = device_system(A, M)
    b = np.ones(n)
    s.rhs().upload(b)
    r = s.solve(rtol=1e-6, max_iter=100000)
    assert r.iterations > 8192
    assert np.linalg.norm(b - M @ s.solution().numpy()) <= 1.1e-6 * np.linalg.norm(b)
    t = s.solve(raise_on_failure=False, rtol=1e-6, max_iter=8200)
    assert t.iterations == 8200 and not t.converged


def test_iteration_limits_and_initial_guess(afem_gpu):
    print("[case] resident limits", flush=True)
    A = afem_gpu
    M = band(3000, [1, 9], shift=0.02)
    x0 = np.random.default_rng(3).normal(size=3000)
    for method in METHODS.values():
        s, keep = device_system(A, M)
        s.rhs().upload(M @ x0)
        s.solution().upload(x0)
        r = s.solve(method=method, rtol=1e-10, use_initial_guess=1)
        assert r.iterations == 0 and r.converged
        assert np.array_equal(s.solution().numpy(), x0)
        r = s.solve(raise_on_failure=False, method=method, rtol=1e-10, max_iter=0)
        assert r.iterations == 0 and not r.converged
        r = s.solve(raise_on_failure=False, method=method, rtol=1e-14, max_iter=5)
        assert r.iterations == 5 and not r.converged
        # solving twice gives the same bits
        s.solve(method=method, rtol=1e-8)
        x = s.solution().numpy()
        s.solve(method=method, rtol=1e-8)
        assert np.array_equal(x, s.solution().numpy())


def test_indefinite_matrix_stops(afem_gpu):
    print("[case] resident indefinite", flush=True)
    A = afem_gpu
    n = 500
    M = sp.diags([np.where(np.arange(n) % 2, 1.0, -1.0)], [0]).tocsr()
    for method in (0, 2):
        s, keep = device_system(A, M)
        s.rhs().upload(np.ones(n))
        r = s.solve(raise_on_failure=False, method=method, rtol=1e-10, max_iter=50)
        s2, keep2 = device_system(A, M)
        s2.rhs().upload(np.ones(n))
        g = s2.solve(raise_on_failure=False, method=method, rtol=1e-10, max_iter=50, spmv_lanes=-1)
        assert (r.converged, r.iterations) == (g.converged, g.iterations)


def test_changed_values_and_pattern(afem_gpu):
    """The kept copy of the matrix follows the values and the pattern."""
    print("[case] resident new values", flush=True)
    A = afem_gpu
    X, C = A.box_mesh(3, 7, 0.15, seed=2)
    m = A.Mesh(3, X, C)
    bsr = A.BSRFormat(m, 1, use_csr=True)
    bsr.compute_sparsity()
    s = A.DoFLinearSystem(X.shape[0])
    on = np.nonzero(X[:, 2] == 0.0)[0].astype(np.int32)
    for k, lam in enumerate((1.0, 7.0)):
        bsr.assemble_laplace(A.DeviceArray.from_numpy(np.full(C.shape[0], lam)), 1.0, s.rhs())
        s.set_bsr(bsr)
        s.apply_dirichlet(A.DIRICHLET_ROW_ELIMINATION, on, 1, 0, 0.0, 0.0)
        s.apply_matrix_transformation()
        s.apply_rhs_transformation()
        for method in (0, 1):
            s.solve(method=method, rtol=1e-10)
            row, col, val, _ = bsr.download()
            M = sp.csr_matrix((val, col, row), shape=(X.shape[0],) * 2)
            b = s.rhs().numpy()
            assert np.linalg.norm(b - M @ s.solution().numpy()) <= 1.01e-10 * np.linalg.norm(b), (k, method)
    M = band(X.shape[0], [3, 11], shift=0.1).tocsr()
    M.sort_indices()
    d = [A.DeviceArray.from_numpy(a) for a in (M.indptr.astype(np.int32)[:-1], M.indices.astype(np.int32), M.data)]
    s.clear_values()
    s.set_csr_values(*d)
    b = np.random.default_rng(0).normal(size=X.shape[0])
    s.rhs().upload(b)
    s.solve(rtol=1e-10)
    assert np.linalg.norm(b - M @ s.solution().numpy()) <= 1.01e-10 * np.linalg.norm(b)


# the flexible method: one and two slices per wave, 16- and 32-bit offsets,
# no off-diagonal pairs in some slices, FP32 and BF16 preconditioner values
FLEX = {"small": (200, [1, 9]), "wave_edge": (4097, [1, 2, 64]), "rows2": (262145, [1, 2, 70]),
        "nine_pairs": (3000, list(range(1, 10))), "far": (70001, [1, 33000, 40001]), "diagonal": (130, [])}


@pytest.mark.parametrize("bf16", [0, 1])
@pytest.mark.parametrize("name", FLEX)
def test_sparse_preconditioner(afem_gpu, name, bf16):
    """M = 2 D^-1 - D^-1 A D^-1 (positive: the spectral radius of D^-1 A is
    below 2 for a diagonally dominant matrix); 1e-6 is above FP32's resolution
    of the residual, where both recurrences take the same iterations."""
    print(f"[case] resident flexible {name} bf16={bf16}", flush=True)
    A = afem_gpu
    n, offsets = FLEX[name]
    M = band(n, offsets, shift=0.05)
    M.sort_indices()
    dinv = 1.0 / M.diagonal()
    rid = np.repeat(np.arange(n), np.diff(M.indptr))
    prec = np.where(M.indices == rid, dinv[rid], -M.data * dinv[rid] * dinv[M.indices]).astype(np.float32)
    b = np.random.default_rng(1).normal(size=n)
    its = {}
    for lanes in (0, -2 if name != "far" else -1):
        s, keep = device_system(A, M)
        s.rhs().upload(b)
        s.set_spai(A.DeviceArray.from_numpy(prec))
        r = s.solve(method=A.SOLVER_FPCG_SPAI, rtol=1e-6, precond_bf16=bf16, spmv_lanes=lanes)
        assert r.converged and not r.fallback
        assert np.linalg.norm(b - M @ s.solution().numpy()) <= 1.01e-6 * np.linalg.norm(b)
        its[lanes] = r.iterations
    a, g = its[0], its[min(its)]
    assert abs(a - g) <= max(3, 0.05 * g), its


def test_sparse_preconditioner_that_is_not_positive_falls_back(afem_gpu):
    print("[case] resident flexible fallback", flush=True)
    A = afem_gpu
    M = band(3000, [1, 9], shift=0.05)
    M.sort_indices()
    rid = np.repeat(np.arange(3000), np.diff(M.indptr))
    prec = np.where(M.indices == rid, -1.0 / M.diagonal()[rid], 0.0).astype(np.float32)
    b = np.random.default_rng(1).normal(size=3000)
    s, keep = device_system(A, M)
    s.rhs().upload(b)
    s.set_spai(A.DeviceArray.from_numpy(prec))
    r = s.solve(method=A.SOLVER_FPCG_SPAI, rtol=1e-8)
    assert r.converged and r.fallback
    assert np.linalg.norm(b - M @ s.solution().numpy()) <= 1.01e-8 * np.linalg.norm(b)


# one launch; two launches (more than 256 systems, a large one among them);
# so many tiny systems that the chunked kernels take over
BATCHES = {"teams": [40, 700, 65, 5000, 1, 64], "two_launches": [70] * 300 + [20000, 3], "chunked": [20] * 2100}


@pytest.mark.parametrize("name", BATCHES)
def test_batches(afem_gpu, name):
    print(f"[case] resident batch {name}", flush=True)
    A = afem_gpu
    parts = [band(n, [1, 7], shift=0.1, seed=k) for k, n in enumerate(BATCHES[name])]
    M = sp.block_diag(parts).tocsr()
    offs = np.concatenate([[0], np.cumsum(BATCHES[name])])
    b = np.random.default_rng(5).normal(size=M.shape[0])
    s, keep = device_system(A, M)
    s.rhs().upload(b)
    bs = A.BatchSolver(s, offs)
    for _ in range(2):
        res, _ = bs.solve(rtol=1e-8)
        r = b - M @ s.solution().numpy()
        for k in range(len(parts)):
            a, e = offs[k], offs[k + 1]
            assert res[k].converged and res[k].relres <= 1e-8
            assert np.linalg.norm(r[a:e]) <= 1.01e-8 * np.linalg.norm(b[a:e]), k
    res, _ = bs.solve(raise_on_failure=False, rtol=1e-13, max_iter=2)
    assert max(q.iterations for q in res) == 2
    # started from the solution: nothing to do
    bs.solve(rtol=1e-8)
    res, _ = bs.solve(rtol=1e-7, use_initial_guess=1)
    assert max(q.iterations for q in res) == 0


def test_batch_with_entries_outside_its_blocks(afem_gpu):
    """Stored zeros that couple two systems: the kernels that read whole vectors take them."""
    print("[case] resident batch couplings", flush=True)
    A = afem_gpu
    M = sp.block_diag([band(300, [1], shift=0.3), band(200, [1], shift=0.3)]).tolil()
    M[299, 300] = M[300, 299] = 1.0
    M = M.tocsr()
    M.sort_indices()
    rid = np.repeat(np.arange(500), np.diff(M.indptr))
    M.data[(rid < 300) != (M.indices < 300)] = 0.0
    b = np.random.default_rng(5).normal(size=500)
    s, keep = device_system(A, M)
    s.rhs().upload(b)
    res, _ = A.BatchSolver(s, [0, 300, 500]).solve(rtol=1e-8)
    r = b - M @ s.solution().numpy()
    assert all(q.converged for q in res)
    assert np.linalg.norm(r[:300]) <= 1.01e-8 * np.linalg.norm(b[:300])
    assert np.linalg.norm(r[300:]) <= 1.01e-8 * np.linalg.norm(b[300:])


@pytest.mark.parametrize("cell,n", [("tri", 5), ("tri", 40), ("tet", 4), ("tet", 13)])
def test_random_numbering(afem_gpu, cell, n):
    """Rows numbered at random are solved in the Morton order that the
    assembly left; the solution comes back in the caller's order, for new
    values too, and for the preconditioner's values."""
    print(f"[case] resident shuffled {cell} {n}", flush=True)
    A = afem_gpu
    dim = 2 if cell == "tri" else 3
    X, C = A.box_mesh(dim, n, 0.15, seed=3)
    order = np.random.default_rng(4).permutation(X.shape[0]).astype(np.int32)
    Y = np.empty_like(X)
    Y[order] = X
    C = np.where(C >= 0, order[np.maximum(C, 0)], -1).astype(np.int32)
    mesh = A.Mesh(dim, Y, C)
    bsr = A.BSRFormat(mesh, 1, use_csr=True)
    bsr.compute_sparsity()
    s = A.DoFLinearSystem(Y.shape[0])
    on = np.nonzero(Y[:, dim - 1] == 0.0)[0].astype(np.int32)
    for lam in (1.0, 3.0):
        bsr.assemble_laplace(A.DeviceArray.from_numpy(np.full(C.shape[0], lam)), 1.0, s.rhs())
        s.set_bsr(bsr)
        s.apply_dirichlet(A.DIRICHLET_ROW_ELIMINATION, on, 1, 0, 0.5, 0.0)
        s.apply_matrix_transformation()
        s.apply_rhs_transformation()
        row, col, val, _ = bsr.download()
        M = sp.csr_matrix((val, col, row), shape=(Y.shape[0],) * 2)
        b = s.rhs().numpy()
        d = M.diagonal()
        rid = np.repeat(np.arange(Y.shape[0]), np.diff(row))
        s.set_spai(A.DeviceArray.from_numpy(np.where(col == rid, 1.0 / d[rid], 0.0).astype(np.float32)))
        for kw in (dict(method=0), dict(method=1), dict(method=3, precond_bf16=0), dict(method=3, precond_bf16=1)):
            A.profile_enable(True)
            A.profile_reset()
            r = s.solve(rtol=1e-8, **kw)
            reordered = A.profile_query("resident_reorder")[0]
            A.profile_reset()
            A.profile_enable(False)
            assert reordered == (1 if Y.shape[0] > 64 else 0), (lam, kw)  # one slice gathers from few lines anyway
            assert np.linalg.norm(b - M @ s.solution().numpy()) <= 1.01e-8 * np.linalg.norm(b), (lam, kw)
            assert r.converged and not r.fallback


def checkerboard_blocks(A, ns):
    """Plane systems with 8x8 checkerboard conductivities from 0.1 to 10, boundary rows eliminated: one union."""
    parts, lams, bnd = [], [], []
    for k, n in enumerate(ns):
        X, C = A.box_mesh(2, n, 0.2, seed=6 + k)
        cell = np.minimum((X[C[:, :3]].mean(axis=1)[:, :2] * 8).astype(int), 7)
        lams.append(np.exp(np.random.default_rng(k).uniform(np.log(0.1), np.log(10.0), 64))[cell[:, 1] * 8 + cell[:, 0]])
        parts.append((X, C))
        bnd.append(np.nonzero((X[:, :2] == 0.0).any(axis=1) | (X[:, :2] == 1.0).any(axis=1))[0])
    X, C, offs = A.union_mesh(parts)
    mesh = A.Mesh(2, X, C)
    bsr = A.BSRFormat(mesh, 1, use_csr=True)
    bsr.compute_sparsity()
    s = A.DoFLinearSystem(X.shape[0])
    bsr.assemble_laplace(A.DeviceArray.from_numpy(np.concatenate(lams)), 1.0, s.rhs())
    s.set_bsr(bsr)
    nodes = np.concatenate([b + o for b, o in zip(bnd, offs)]).astype(np.int32)
    s.apply_dirichlet(A.DIRICHLET_ROW_ELIMINATION, nodes, 1, 0, 0.0, 0.0)
    s.apply_matrix_transformation()
    s.apply_rhs_transformation()
    return s, offs, (mesh, bsr)


def test_mixed_precision_takes_no_more_iterations_than_fp64(afem_gpu):
    """Hard coefficients: the mixed solver's rounding neither delays it (2 %,
    measured 0.4 %) nor leaves more error than FP64 PCG's stopping residual
    does (ten times it: at the same residual the error moves by a few times
    with the last iterations' rounding)."""
    print("[case] mixed against FP64 iterations", flush=True)
    A = afem_gpu
    for n in (197, 250, 320):
        s, offs, keep = checkerboard_blocks(A, [n])
        s.solve(method=METHODS["fp64"], rtol=1e-11, max_iter=20000)
        x = s.solution().numpy()
        err, its = {}, {}
        for m in ("fp64", "mixed"):
            its[m] = s.solve(method=METHODS[m], rtol=1e-8, max_iter=20000).iterations
            err[m] = np.linalg.norm(s.solution().numpy() - x) / np.linalg.norm(x)
        print(f"[result] n={n} {its} {err}", flush=True)
        assert its["mixed"] <= 1.02 * its["fp64"] + 3
        assert err["mixed"] <= 10 * err["fp64"]


def test_batch_takes_no_more_iterations_than_the_chunked_kernels(afem_gpu):
    """What a caller's max_iter allowed them is enough for the default solve."""
    print("[case] batch against chunked iterations", flush=True)
    A = afem_gpu
    s, offs, keep = checkerboard_blocks(A, [60, 197, 320, 250])
    bs = A.BatchSolver(s, offs)
    res, _ = bs.solve(rtol=1e-8, max_iter=20000)
    bs.set_tiles(1, 1)
    ref, _ = bs.solve(rtol=1e-8, max_iter=20000)
    its = [(a.iterations, g.iterations) for a, g in zip(res, ref)]
    print(f"[result] {its}", flush=True)
    assert all(a <= 1.02 * g + 3 for a, g in its), its


@pytest.mark.parametrize("offsets", [[1, 2, 70], [1, 33000, 40001]], ids=["near", "far"])
def test_spmv_format_after_a_solve(afem_gpu, offsets):
    """The format that is reported is the one that the products use."""
    print(f"[case] spmv format after a solve {offsets}", flush=True)
    A = afem_gpu
    n = 70001
    M = band(n, offsets, shift=0.3)
    s, keep = device_system(A, M)
    b = np.random.default_rng(1).normal(size=n)
    s.rhs().upload(b)
    assert s.spmv_format() is None
    s.solve(rtol=1e-8)
    x = s.solution().numpy()
    fmt, tuning = s.spmv_format(), s.spmv_tuning()
    assert fmt is not None
    assert (tuning[0] != (0, 0)) == fmt[0].startswith("sell16"), (fmt, tuning)
    y = A.DeviceArray(n, np.float64)
    s.spmv(s.rhs(), y)
    assert np.abs(y.numpy() - M @ b).max() <= 1e-12 * np.abs(M @ b).max()
    assert s.spmv_format() == fmt and s.spmv_tuning() == tuning
    s.solve(rtol=1e-8)
    assert np.array_equal(s.solution().numpy(), x)
