"""Without strain the internal forces and the material derivatives of the VJP
vanish to the last bit (F = I, ln J = 0, b = I exactly), on cells whose edge
lengths are no machine numbers, so a load step without load converges: its
residual is zero, and no rounding of terms that cancel is left to be iterated
on.
"""
import numpy as np
import pytest

import lsmf

pytestmark = pytest.mark.gpu

SHEAR = np.array([[1.0, 0.3, -0.2], [0.1, 0.8, 0.25], [-0.15, 0.2, 1.1]])


@pytest.mark.parametrize("dim,p,n", [(3, 2, [7, 3, 5]), (3, 2, [1, 1, 1]), (3, 2, [10, 2, 3]), (3, 4, [3, 2, 1]),
                                     (2, 2, [7, 3])], ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("geometry", ["box", "sheared", "cook"])
@pytest.mark.parametrize("caching", ["tensor4", "scalar"])
def test_no_strain_no_force(dim, p, n, geometry, caching, device):
    import torch
    print(f"[no strain] dim={dim} p={p} n={n} {geometry} {caching}", flush=True)
    mesh = lsmf.Mesh(dim, p, n, geometry="cook" if geometry == "cook" else "box")
    if geometry == "sheared":
        mesh.coords = np.ascontiguousarray(mesh.coords @ SHEAR[:dim, :dim].T)
    rng = np.random.default_rng(1)
    op = lsmf.NeoHookOperator(mesh, caching=caching)
    op.set_material(1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells))
    op.set_linearization(torch.zeros(mesh.n_dofs, dtype=torch.float64, device=device))
    r = torch.full((mesh.n_dofs,), float("nan"), dtype=torch.float64, device=device)
    op.residual(r)
    du = torch.full_like(r, float("nan"))
    dmu, dlam = (torch.full((mesh.n_cells,), float("nan"), dtype=torch.float64, device=device) for _ in range(2))
    op.residual_vjp(torch.tensor(rng.standard_normal(mesh.n_dofs), device=device), du, dmu, dlam)
    assert float(r.abs().max()) == 0.0
    assert float(dmu.abs().max()) == 0.0 and float(dlam.abs().max()) == 0.0


@pytest.mark.parametrize("coarse", [[3, 2, 1], [2, 2, 2]], ids=str)
def test_step_without_load_converges(coarse, device):
    print(f"[no load] {coarse}", flush=True)
    o = lsmf.solver_options(dim=3, degree=2, n_q_1d=3, n_cells_coarse=coarse, n_levels=2, caching="tensor4",
                            mg_caching="tensor4", mg_precision="fp64", dt=1.0, t_end=1.0,
                            dirichlet={0: ([0, 1, 2], [0.0] * 3), 1: ([0], [0.0])})
    n_cells = 8 * int(np.prod(coarse))
    s = lsmf.Solver(o, np.full(n_cells, 1.0), np.full(n_cells, 1.7))
    stats = s.run()
    assert len(stats) == 1 and stats[0]["residual_0"] == 0.0
    assert np.abs(s.solution()).max() == 0.0
