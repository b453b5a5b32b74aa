"""Q2 products on affine cells on both sides of the tile counts at which their
kernel changes (16 and 512 wide tiles of 9x2x1 cells), against the oracle: FP64
to 1e-12, FP32 to 2e-5 (max-norm), the tolerances of the operator's other parity
tests; one launch over all tiles and one per colour give the same bits.
"""
import numpy as np
import pytest

import lsmf
import oracle

pytestmark = pytest.mark.gpu

SHEAR = np.array([[1.0, 0.3, -0.2], [0.1, 0.8, 0.25], [-0.15, 0.2, 1.1]])
# tiles: 16, 17, 512, 513
MESHES = [[9, 7, 4], [8, 2, 17], [18, 15, 32], [27, 17, 19]]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-5)])
@pytest.mark.parametrize("n", MESHES, ids=str)
def test_products_about_the_rules(n, precision, tol, device):
    import torch
    print(f"[q2 rules] {n} {precision}", flush=True)
    mesh = lsmf.Mesh(3, 2, n)
    mesh.coords = np.ascontiguousarray(mesh.coords @ SHEAR.T)
    rng = np.random.default_rng(3)
    mu, lam = 1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells)
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.02, 7)
    cons = mesh.constrained_mask({0: [0, 1, 2], 1: [0]})
    ref = oracle.OracleOperator(3, 2, mesh.cell_nodes, mesh.coords, cons, caching="tensor4")
    ref.set_material(mu, lam)
    ref.set_linearization(u)
    ref.cache()
    v = rng.standard_normal(mesh.n_dofs).astype(np.float32).astype(np.float64)
    expect, diag = ref.vmult(v), ref.diagonal()
    op = lsmf.NeoHookOperator(mesh, precision=precision, caching="tensor4", constrained=cons)
    op.set_material(mu, lam)
    op.set_linearization(torch.tensor(u, device=device))
    op.cache()
    x = torch.tensor(v, device=device).to(op.dtype)
    y, z = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    op.vmult(y, x)
    torch.cuda.synchronize()
    op.vmult(z, x, stream=torch.cuda.Stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(y, z)
    batch = torch.full((2, x.numel()), float("nan"), device=device, dtype=op.dtype)
    op.vmult_batched(batch, torch.stack([x, x]))
    assert torch.equal(batch[0], y) and torch.equal(batch[1], y)
    assert np.abs(y.double().cpu().numpy() - expect).max() < tol * np.abs(expect).max()
    op.compute_diagonal()
    assert np.abs(op.diagonal().double().cpu().numpy() - diag).max() < tol * np.abs(diag).max()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-13), ("fp32", 1e-5)])
@pytest.mark.parametrize("caching", ["tensor4", "scalar"])
@pytest.mark.parametrize("n", [[1, 1, 1], [10, 3, 5], [8, 2, 17]], ids=str)
@pytest.mark.parametrize("geometry", ["sheared", "cook"])
def test_phase_masks(n, geometry, caching, precision, tol, device):
    """products without the tangent, and without the sums, against those of the
    cells layout, one launch and coloured launches alike"""
    import torch
    print(f"[phases] {n} {geometry} {caching} {precision}", flush=True)
    mesh = lsmf.Mesh(3, 2, n, geometry="cook" if geometry == "cook" else "box")
    if geometry == "sheared":
        mesh.coords = np.ascontiguousarray(mesh.coords @ SHEAR.T)
    rng = np.random.default_rng(3)
    mu, lam = 1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells)
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.02, 7)
    cons = mesh.constrained_mask({0: [0, 1, 2], 1: [0]})
    ops = []
    for layout in ("auto", "cells"):
        op = lsmf.NeoHookOperator(mesh, precision=precision, caching=caching, constrained=cons, layout=layout)
        op.set_material(mu, lam)
        op.set_linearization(torch.tensor(u, device=device))
        op.cache()
        ops.append(op)
    x = torch.tensor(rng.standard_normal(mesh.n_dofs), device=device).to(ops[0].dtype)
    for mask in ("rw", "rwsf", "default"):
        y, z, w = (torch.full_like(x, float("nan")) for _ in range(3))
        ops[1].vmult(w, x, mask=mask)
        ops[0].vmult(y, x, mask=mask)
        torch.cuda.synchronize()
        ops[0].vmult(z, x, mask=mask, stream=torch.cuda.Stream().cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(y, z), mask
        assert float((y - w).abs().max()) < tol * float(w.abs().max()), mask
