"""Whether the cells are taken as affine depends on each cell's own vertices:
not on a node that no cell has, however far away, nor on how large the rest of
the mesh is.  Products against the oracle, FP64 to 1e-12 and FP32 to 2e-5
(max-norm), the tolerances of the operator's other parity tests.
"""
import numpy as np
import pytest

import lsmf
import oracle

pytestmark = pytest.mark.gpu


def product(mesh, mu, lam, u, v, caching, precision, device):
    import torch
    op = lsmf.NeoHookOperator(mesh, precision=precision, caching=caching)
    op.set_material(mu, lam)
    op.set_linearization(torch.tensor(u, device=device))
    op.cache()
    x = torch.tensor(v, device=device).to(op.dtype)
    y = torch.full_like(x, float("nan"))
    op.vmult(y, x)
    return y.double().cpu().numpy()


def expected(mesh, mu, lam, u, v):
    ref = oracle.OracleOperator(mesh.dim, mesh.degree, mesh.cell_nodes, mesh.coords, np.zeros(mesh.n_dofs, np.uint8),
                                caching="tensor4")
    ref.set_material(mu, lam)
    ref.set_linearization(u)
    ref.cache()
    return ref.vmult(v)


@pytest.mark.parametrize("dim,p,n", [(2, 2, [5, 3]), (3, 1, [4, 3, 2]), (3, 2, [4, 3, 2]), (3, 4, [2, 2, 1])],
                         ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("caching,precision,tol", [("tensor4", "fp64", 1e-12), ("tensor4", "fp32", 2e-5),
                                                   ("scalar", "fp64", 1e-12)])
@pytest.mark.parametrize("far", [1e14, 1e200])
def test_unreferenced_node_far_away(dim, p, n, caching, precision, tol, far, device):
    print(f"[affine rule] dim={dim} p={p} {caching} {precision} {far}", flush=True)
    mesh = lsmf.Mesh(dim, p, n, geometry="cook")  # bilinear cells
    mesh.coords = np.ascontiguousarray(np.vstack([mesh.coords, np.full((1, dim), far)]))
    mesh.n_nodes += 1
    rng = np.random.default_rng(2)
    mu, lam = 1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells)
    u, _ = lsmf.smooth_displacement(mesh.coords[:-1], 0.02, 7)
    u = np.concatenate([u, np.zeros(dim)])
    v = rng.standard_normal(mesh.n_dofs).astype(np.float32).astype(np.float64)
    e = expected(mesh, mu, lam, u, v)
    y = product(mesh, mu, lam, u, v, caching, precision, device)
    assert np.abs(y - e).max() < tol * np.abs(e).max()


@pytest.mark.parametrize("caching", ["tensor4", "scalar"])
def test_small_cells_of_a_large_mesh(caching, device):
    """cells of size 1e-7 whose bilinear part is 1e-8 of it, 1e-15, in a mesh
    that reaches x = 1: it counts at the nodes of those cells"""
    h = 1e-7
    mesh = lsmf.Mesh(3, 2, [4, 3, 2])
    X = mesh.coords.copy()
    X[:, 0] += 1e-8 * X[:, 1] * X[:, 2]
    X *= h
    last = mesh.coords[:, 0] > 0.76  # the last layer of cells is stretched to x = 1
    X[last, 0] += 1.0
    mid = np.abs(mesh.coords[:, 0] - 0.875) < 1e-12
    X[mid, 0] -= 0.5
    mesh.coords = np.ascontiguousarray(X)
    rng = np.random.default_rng(2)
    mu, lam = 1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells)
    u = 0.01 * h * np.sin(np.arange(mesh.n_dofs))
    v = rng.standard_normal(mesh.n_dofs)
    small = np.repeat(X[:, 0] < 0.7 * h, 3)  # nodes of the small cells only
    e = expected(mesh, mu, lam, u, v)[small]
    y = product(mesh, mu, lam, u, v, caching, "fp64", device)[small]
    assert np.abs(y - e).max() < 1e-12 * np.abs(e).max()
