"""The compact form of the tensor2 / tensor4 products (K, c dw per point, the
rest per affine cell or per point) against the oracle's stored tensors, on
parallelepiped cells (affine, J_ref not diagonal), on the Cook geometry
(bilinear cells) and over the formulation switch, at mesh sizes that leave
tiles full, ragged and nearly empty.  FP64 to 1e-12, FP32 to 2e-5 (max-norm),
the tolerances of the operator's other parity tests.
"""
import numpy as np
import pytest

import lsmf
import oracle

pytestmark = pytest.mark.gpu

SHEAR = np.array([[1.0, 0.3, -0.2], [0.1, 0.8, 0.25], [-0.15, 0.2, 1.1]])


def rel(a, b):
    return float(np.abs(a - b).max() / np.abs(b).max())


def problem(dim, p, n, geometry):
    mesh = lsmf.Mesh(dim, p, n, geometry="cook" if geometry == "cook" else "box")
    if geometry == "sheared":
        mesh.coords = np.ascontiguousarray(mesh.coords @ SHEAR[:dim, :dim].T)
    rng = np.random.default_rng(3)
    mu, lam = 1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells)
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.02, 7)
    cons = mesh.constrained_mask({0: list(range(dim)), 1: [0]})
    return mesh, mu, lam, u, cons


def oracle_op(mesh, mu, lam, u, cons, caching, formulation=1):
    ref = oracle.OracleOperator(mesh.dim, mesh.degree, mesh.cell_nodes, mesh.coords, cons, caching=caching,
                                formulation=formulation)
    ref.set_material(mu, lam)
    ref.set_linearization(u)
    ref.cache()
    return ref


@pytest.mark.parametrize("geometry", ["sheared", "cook"])
@pytest.mark.parametrize("dim,p,n", [(2, 1, [9, 8]), (2, 2, [8, 5]), (2, 4, [6, 3]), (3, 1, [5, 4, 3]),
                                     (3, 2, [1, 1, 1]), (3, 2, [9, 2, 1]), (3, 2, [15, 3, 5]), (3, 4, [1, 1, 1]),
                                     (3, 4, [5, 3, 2])],
                         ids=lambda v: str(v).replace(" ", ""))
def test_compact_products_match_oracle(dim, p, n, geometry, device):
    import torch
    print(f"[compact] dim={dim} p={p} n={n} {geometry}", flush=True)
    mesh, mu, lam, u, cons = problem(dim, p, n, geometry)
    ref = oracle_op(mesh, mu, lam, u, cons, "tensor4")
    rng = np.random.default_rng(4)
    v, w = (rng.standard_normal(mesh.n_dofs).astype(np.float32).astype(np.float64) for _ in range(2))
    expect, plain, diag = ref.vmult(v), ref.vmult(v, plain=True), ref.diagonal()
    for layout in ("auto", "cells"):
        for prec, tol in (("fp64", 1e-12), ("fp32", 2e-5)):
            op = lsmf.NeoHookOperator(mesh, precision=prec, caching="tensor4", constrained=cons, layout=layout)
            op.set_material(mu, lam)
            op.set_linearization(torch.tensor(u, device=device))
            op.cache()
            src = torch.tensor(v, device=device, dtype=op.dtype)
            y = torch.full_like(src, np.nan)
            op.vmult(y, src)
            assert rel(y.cpu().double().numpy(), expect) < tol, (layout, prec)
            y = torch.tensor(w, device=device, dtype=op.dtype)
            op.vmult_add(y, src)
            assert rel(y.cpu().double().numpy(), w + expect) < tol, (layout, prec)
            y = torch.full_like(src, np.nan)
            op.vmult(y, src, mask="plain")
            assert rel(y.cpu().double().numpy(), plain) < tol, (layout, prec)
            batch = torch.stack([src, 2 * src, -src])
            out = torch.full_like(batch, np.nan)
            op.vmult_batched(out, batch)
            op.vmult(y, src)
            assert torch.equal(out[0], y) and torch.equal(out[1], 2 * y) and torch.equal(out[2], -y)
            op.compute_diagonal()
            assert rel(op.diagonal().cpu().double().numpy(), diag) < tol, (layout, prec)


def test_formulation_switch_changes_the_cached_values(device):
    import torch
    mesh, mu, lam, u, cons = problem(3, 2, [4, 3, 2], "sheared")
    v = np.random.default_rng(4).standard_normal(mesh.n_dofs)
    op = lsmf.NeoHookOperator(mesh, caching="tensor4", constrained=cons)
    op.set_material(mu, lam)
    op.set_linearization(torch.tensor(u, device=device))
    src = torch.tensor(v, device=device)
    y = torch.empty_like(src)
    bytes_of = {}
    for formulation in (1, 0, 1, 0):
        lsmf._check(lsmf._lib.lsmf_set_formulation(op._h, formulation))
        with pytest.raises(lsmf.LsmfError):
            op.vmult(y, src)  # the cache is of the other formulation
        op.cache()
        op.vmult(y, src)
        expect = oracle_op(mesh, mu, lam, u, cons, "tensor4", formulation).vmult(v)
        assert rel(y.cpu().numpy(), expect) < 1e-12, formulation
        assert bytes_of.setdefault(formulation, op.memory_consumption()) == op.memory_consumption()


def test_products_keep_the_cached_state(device):
    """a product after cache() uses the state that was cached: the next
    linearisation state may be set (on another stream) while it runs, and no
    product runs between set_linearization and cache()"""
    import torch
    mesh, mu, lam, u, cons = problem(3, 2, [19, 9, 9], "sheared")
    x = torch.tensor(np.random.default_rng(1).standard_normal(mesh.n_dofs), device=device)
    op = lsmf.NeoHookOperator(mesh, caching="tensor4", constrained=cons)
    op.set_material(mu, lam)
    op.set_linearization(torch.tensor(u, device=device))
    op.cache()
    expect = oracle_op(mesh, mu, lam, u, cons, "tensor4").vmult(x.cpu().numpy())
    other, ys = torch.cuda.Stream(), [torch.empty_like(x) for _ in range(20)]
    zero = torch.zeros_like(x)
    torch.cuda.synchronize()
    for y in ys:
        op.vmult(y, x)
    op.set_linearization(zero, stream=other.cuda_stream)
    torch.cuda.synchronize()
    for y in ys:
        assert rel(y.cpu().numpy(), expect) < 1e-12
    with pytest.raises(lsmf.LsmfError):
        op.vmult(ys[0], x)
    op.cache()
    op.vmult(ys[0], x)
    assert rel(ys[0].cpu().numpy(), oracle_op(mesh, mu, lam, 0 * u, cons, "tensor4").vmult(x.cpu().numpy())) < 1e-12


@pytest.mark.parametrize("geometry", ["sheared", "cook"])
@pytest.mark.parametrize("n", [[1, 1, 1], [9, 2, 1], [10, 3, 5], [19, 5, 2]], ids=str)
def test_residual_and_vjp(n, geometry, device):
    """internal forces against the oracle; du of the VJP is -A w (oracle), and
    w . R is linear in each cell's mu and lambda with coefficients dmu, dlambda"""
    import torch
    print(f"[residual] n={n} {geometry}", flush=True)
    mesh, mu, lam, u, cons = problem(3, 2, n, geometry)
    op = lsmf.NeoHookOperator(mesh, caching="tensor4", constrained=cons)
    op.set_linearization(torch.tensor(u, device=device))

    def residual(m, l):
        op.set_material(m, l)
        r = torch.full((mesh.n_dofs,), float("nan"), dtype=torch.float64, device=device)
        op.residual(r)
        return r.cpu().numpy()

    rng = np.random.default_rng(6)
    w, hm, hl = rng.standard_normal(mesh.n_dofs), rng.random(mesh.n_cells), rng.random(mesh.n_cells)
    base, more_mu, more_lam = residual(mu, lam), residual(mu + hm, lam), residual(mu, lam + hl)
    ref = oracle_op(mesh, mu, lam, u, cons, "tensor4")
    expect = ref.residual()
    assert np.abs(base - expect).max() < 1e-12 * np.abs(expect).max()
    op.set_material(mu, lam)
    du = torch.full((mesh.n_dofs,), float("nan"), dtype=torch.float64, device=device)
    dmu, dlam = (torch.full((mesh.n_cells,), float("nan"), dtype=torch.float64, device=device) for _ in range(2))
    op.residual_vjp(torch.tensor(w, device=device), du, dmu, dlam)
    assert rel(du.cpu().numpy(), -ref.vmult(w, plain=True)) < 1e-12
    for h, other, grad in ((hm, more_mu, dmu), (hl, more_lam, dlam)):
        terms = w * (other - base)  # rounding of the difference of two residuals
        assert abs(float(h @ grad.cpu().numpy()) - terms.sum()) < 1e-12 * np.abs(w * base).sum()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-5)])
@pytest.mark.parametrize("n", [[1, 1, 1], [9, 1, 1], [10, 3, 5], [19, 2, 2]], ids=str)
@pytest.mark.parametrize("geometry", ["sheared", "cook"])
def test_scalar_products(n, geometry, precision, tol, device):
    """scalar caching on affine cells (planes and columns) and on bilinear ones,
    formulation 1, then 0, then 1 again, against the oracle"""
    import torch
    print(f"[scalar] n={n} {geometry} {precision}", flush=True)
    mesh, mu, lam, u, cons = problem(3, 2, n, geometry)
    op = lsmf.NeoHookOperator(mesh, precision=precision, caching="scalar", constrained=cons)
    op.set_material(mu, lam)
    v = np.random.default_rng(4).standard_normal(mesh.n_dofs).astype(np.float32).astype(np.float64)
    for formulation in (1, 0, 1):
        assert lsmf._lib.lsmf_set_formulation(op._h, formulation) == lsmf.LSMF_OK
        op.set_linearization(torch.tensor(u, device=device))
        op.cache()
        expect = oracle_op(mesh, mu, lam, u, cons, "scalar", formulation).vmult(v)
        y = torch.full((mesh.n_dofs,), float("nan"), dtype=op.dtype, device=device)
        op.vmult(y, torch.tensor(v, device=device).to(op.dtype))
        assert rel(y.double().cpu().numpy(), expect) < tol, formulation
