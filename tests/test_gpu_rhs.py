"""Right-hand sides summed per node from per-cell terms, against the oracle.

The sums have up to a few hundred FP64 terms of one sign per node, so any
order of addition agrees to well below 1e-13 of the largest entry.
"""

import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu


def fan(dim, k):
    """k cells around one node (triangles) or one edge (tetrahedra): lists
    longer than one round of lanes."""
    a = 2 * np.pi * np.arange(k) / k
    ring = np.stack([np.cos(a), np.sin(a), np.zeros(k)], axis=1)
    nxt = (np.arange(k) + 1) % k
    if dim == 2:
        X = np.concatenate([[[0.1, 0.05, 0.0]], ring])
        C = np.stack([np.zeros(k, int), 1 + np.arange(k), 1 + nxt, np.full(k, -1)], axis=1)
    else:
        X = np.concatenate([[[0.1, 0.05, -1.0], [0.0, 0.1, 1.0]], ring])
        C = np.stack([np.zeros(k, int), 2 + np.arange(k), 2 + nxt, np.ones(k, int)], axis=1)
    return X, C.astype(np.int32)


def shuffled(X, C, seed):
    order = np.random.default_rng(seed).permutation(X.shape[0]).astype(np.int32)
    Y = np.empty_like(X)
    Y[order] = X
    return Y, np.where(C >= 0, order[np.maximum(C, 0)], -1).astype(np.int32)


def meshes(A, name):
    if name.startswith("fan"):
        dim, k = int(name[3]), int(name[5:])
        return (dim,) + fan(dim, k)
    cell, n = name.split("_")
    dim = 2 if cell in ("tri", "quad") else 3
    X, C = A.box_mesh(dim, int(n), 0.15, seed=4) if cell in ("tri", "tet") else A.box_mesh_q1(dim, int(n), 0.15, seed=4)
    return (dim,) + shuffled(X, C, 9)


@pytest.mark.parametrize("name", ["fan2_3", "fan2_60", "fan3_3", "fan3_8", "fan3_25", "fan3_49", "tri_1", "tri_17",
                                  "tet_1", "tet_7", "quad_1", "quad_13", "hexa_1", "hexa_6"])
def test_sources_and_mass(afem_gpu, name):
    A = afem_gpu
    print(f"[case] rhs {name}", flush=True)
    dim, X, C = meshes(A, name)
    npc = 8 if C.shape[1] == 8 else 4 if name.startswith(("quad", "tet", "fan3", "hexa")) else 3
    m = A.Mesh(dim, X, C, npc=npc)
    N = X.shape[0]
    rng = np.random.default_rng(0)
    u, scale = rng.normal(size=N), rng.uniform(0.5, 2.0, C.shape[0])
    # the source overwrites, the mass term adds, both into one component of two
    r0 = rng.normal(size=2 * N)
    got = A.DeviceArray.from_numpy(r0)
    sc = A.DeviceArray.from_numpy(scale)
    A.check(A.lib().afem_rhs_constant_source(m.h, 1.7, sc.c, 2, 1, got.c))
    ref = O.rhs_constant_source(dim, X, C, npc, 1.7, cell_scale=scale)
    out = got.numpy()
    assert np.array_equal(out[0::2], r0[0::2])
    assert np.abs(out[1::2] - ref).max() <= 1e-13 * np.abs(ref).max()
    A.rhs_mass_field(m, A.DeviceArray.from_numpy(u), 3.0, got, nb_dof=2, dof_index=0)
    ref = O.rhs_mass_field(X, C, npc, u, 3.0, rhs=r0[0::2].copy(), dim=dim)
    out2 = got.numpy()
    assert np.array_equal(out2[1::2], out[1::2])
    # r0 of size 1 joins the sum: its rounding counts too
    assert np.abs(out2[0::2] - ref).max() <= 1e-13 * max(1.0, np.abs(ref).max())
    if dim == 3 and npc == 4:
        f = np.array([0.3, -2.0, 1.0])
        got = A.DeviceArray.from_numpy(np.zeros(3 * N))
        A.check(A.lib().afem_rhs_body_force(m.h, A._ptr(f), got.c))
        ref = O.rhs_body_force(X, C, f)
        assert np.abs(got.numpy() - ref).max() <= 1e-13 * np.abs(ref).max()


@pytest.mark.parametrize("name", ["tri_5", "tet_4", "quad_4", "hexa_3"])
def test_nodes_without_cells(afem_gpu, name):
    """Unused nodes get nothing, also where the field is not a number."""
    A = afem_gpu
    print(f"[case] rhs unused nodes {name}", flush=True)
    dim, X, C = meshes(A, name)
    npc = 8 if C.shape[1] == 8 else 3 if name.startswith("tri") else 4
    N = X.shape[0]
    Y = np.concatenate([[[9.0, 9.0, 0.0]], X, np.full((2, 3), 7.0) * [1.0, 1.0, 0.0]])
    m = A.Mesh(dim, Y, np.where(C >= 0, C + 1, -1).astype(np.int32), npc=npc)
    rng = np.random.default_rng(0)
    u, r0 = rng.normal(size=N), rng.normal(size=N + 3)
    field = np.concatenate([[np.nan], u, [np.inf, -np.inf]])
    got = A.DeviceArray.from_numpy(r0)
    A.rhs_mass_field(m, A.DeviceArray.from_numpy(field), 3.0, got)
    ref = O.rhs_mass_field(X, C, npc, u, 3.0, rhs=r0[1:-2].copy(), dim=dim)
    out = got.numpy()
    assert np.array_equal(out[[0, -2, -1]], r0[[0, -2, -1]])
    assert np.abs(out[1:-2] - ref).max() <= 1e-13 * max(1.0, np.abs(ref).max())
