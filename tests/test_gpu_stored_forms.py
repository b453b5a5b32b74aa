"""The stored tensors, which only curved meshes, formulation 0 and tensor4_ns
read, against the compact form of the same tangent, which all other tensor2,
tensor4 and affine scalar products share.

  * full sizes: the compact form against tensor4_ns, another kernel on other
    cached values (dP/dF and J_ref^-1), FP64 to 1e-12 (max-norm)
  * curved meshes whose wide tiles are ragged in every direction: products and
    diagonal of tensor2 and tensor4 against the oracle, FP64 to 1e-12, FP32 to
    2e-5, the tolerances of the operator's other parity tests
"""
import numpy as np
import pytest

import curved_mesh
import lsmf
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,caching", [(3, "tensor4"), (2, "tensor4"), (4, "tensor2"), (3, "scalar")])
def test_full_size_against_tensor4_ns(cfg, caching, device):
    import torch
    print(f"[stored forms] config {cfg} {caching}", flush=True)
    mesh, mu, lam = lsmf.build_config_mesh(cfg)
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.02, 5)
    cons = mesh.constrained_mask({0: [0, 1, 2], 1: [0]})
    x = torch.tensor(np.random.default_rng(6).standard_normal(mesh.n_dofs), device=device)
    out, diag = [], []
    for form in (caching, "tensor4_ns"):
        op = lsmf.NeoHookOperator(mesh, caching=form, constrained=cons)
        op.set_material(mu, lam)
        op.set_linearization(torch.tensor(u, device=device))
        op.cache()
        y = torch.full_like(x, float("nan"))
        op.vmult(y, x)
        op.compute_diagonal()
        out.append(y)
        diag.append(op.diagonal())
        del op
        torch.cuda.empty_cache()
    assert float((out[0] - out[1]).abs().max()) < 1e-12 * float(out[1].abs().max())
    assert float((diag[0] - diag[1]).abs().max()) < 1e-12 * float(diag[1].abs().max())


@pytest.mark.parametrize("p,n", [(2, [10, 3, 2]), (2, [19, 5, 3]), (4, [5, 3, 2]), (4, [9, 2, 1])],
                         ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("caching", ["tensor2", "tensor4"])
def test_curved_ragged_tiles_match_oracle(p, n, caching, device):
    import torch
    print(f"[stored forms] curved Q{p} {n} {caching}", flush=True)
    mesh = curved_mesh.annulus(3, p, n)
    rng = np.random.default_rng(4)
    mu, lam = 1.0 + rng.random(mesh.n_cells), 1.5 + rng.random(mesh.n_cells)
    u = (0.02 * np.sin(2.0 * mesh.coords @ np.arange(1, 4))[:, None] * np.linspace(1.0, 0.5, 3)).reshape(-1)
    cons = mesh.constrained_mask({2: [0, 1, 2]})
    ref = oracle.OracleOperator(3, p, mesh.cell_nodes, mesh.coords, cons, caching=caching)
    ref.set_material(mu, lam)
    ref.set_linearization(u)
    ref.cache()
    v, w = (rng.standard_normal(mesh.n_dofs).astype(np.float32).astype(np.float64) for _ in range(2))
    expect, plain, diag = ref.vmult(v), ref.vmult(v, plain=True), ref.diagonal()
    other = torch.cuda.Stream()
    for prec, tol in (("fp64", 1e-12), ("fp32", 2e-5)):
        op = lsmf.NeoHookOperator(mesh, precision=prec, caching=caching, constrained=cons)
        op.set_material(mu, lam)
        op.set_linearization(torch.tensor(u, device=device))
        op.cache()
        x = torch.tensor(v, device=device).to(op.dtype)
        for stream in (None, other.cuda_stream):  # one launch over all tiles, one per colour
            for kw, e in (({}, expect), ({"mask": "plain"}, plain), ({"add": True}, w + expect)):
                y = torch.tensor(w, device=device).to(op.dtype) if kw.get("add") else torch.full_like(x, float("nan"))
                torch.cuda.synchronize()
                op.vmult(y, x, stream=stream, **kw)
                torch.cuda.synchronize()
                assert np.abs(y.double().cpu().numpy() - e).max() < tol * np.abs(e).max(), (prec, stream, kw)
        op.compute_diagonal()
        assert np.abs(op.diagonal().double().cpu().numpy() - diag).max() < tol * np.abs(diag).max(), prec
