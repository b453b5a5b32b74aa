"""Products recorded in a graph stay valid over set_formulation: a replay gives
the product of what cache() cached last, in either formulation, though the two
keep different values per point; until then it gives the one before.  Replays
alternate with eager products, other allocations and synchronizations, and are
compared with the eager products (same bits) and with the oracle (FP64 to 1e-12,
FP32 to 2e-5, max-norm, as the operator's other parity tests).
"""
import numpy as np
import pytest

import hanging_mesh
import lsmf
import oracle

pytestmark = pytest.mark.gpu

SHEAR = np.array([[1.0, 0.3, -0.2], [0.1, 0.8, 0.25], [-0.15, 0.2, 1.1]])
CASES = [(3, 2, [10, 3, 4], "sheared", "auto"), (3, 2, [10, 3, 4], "cook", "auto"), (3, 2, [3, 2, 2], "box", "cells"),
         (3, 4, [5, 2, 1], "sheared", "auto"), (3, 4, [2, 2, 1], "cook", "auto"), (3, 1, [5, 4, 3], "box", "auto"),
         (2, 2, [9, 7], "cook", "auto"), (2, 4, [5, 3], "sheared", "auto"), (3, 2, None, "hanging", "cells")]


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 2e-5)])
@pytest.mark.parametrize("dim,p,n,geometry,layout", CASES, ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("first", [1, 0])
def test_replays_follow_the_cache(dim, p, n, geometry, layout, precision, tol, first, device):
    import torch
    print(f"[recorded] dim={dim} p={p} n={n} {geometry} {layout} {precision} {first}", flush=True)
    nc = None
    if geometry == "hanging":
        mesh, nc = hanging_mesh.build(dim, p)
    else:
        mesh = lsmf.Mesh(dim, p, n, geometry="cook" if geometry == "cook" else "box")
    if geometry == "sheared":
        mesh.coords = np.ascontiguousarray(mesh.coords @ SHEAR[:dim, :dim].T)
    rng = np.random.default_rng(3)
    mu, lam = 1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells)
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.02, 7)
    if nc is not None:
        u = hanging_mesh.constraint_matrix(mesh, nc) @ u  # a displacement of that mesh is continuous
    v = rng.standard_normal(mesh.n_dofs).astype(np.float32).astype(np.float64)
    op = lsmf.NeoHookOperator(mesh, precision=precision, caching="tensor4", layout=layout, formulation=first,
                              use_mesh_colouring=geometry != "hanging", node_constraints=nc)
    op.set_material(mu, lam)
    op.set_linearization(torch.tensor(u, device=device))
    op.cache()
    x = torch.tensor(v, device=device).to(op.dtype)
    start = torch.linspace(-1, 1, x.numel(), device=device, dtype=op.dtype)
    batch = torch.stack([x, 2 * x])
    y, z, w = torch.empty_like(x), torch.empty_like(x), torch.empty_like(batch)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.vmult(y, x)
        z.copy_(start)
        op.vmult_add(z, x)
        op.vmult_batched(w, batch)

    def replay():
        for t in (y, z, w):
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        return y.clone(), z.clone(), w.clone()

    def eager():
        a, b, c = torch.full_like(x, float("nan")), start.clone(), torch.full_like(batch, float("nan"))
        op.vmult(a, x)
        op.vmult_add(b, x)
        op.vmult_batched(c, batch)
        torch.cuda.synchronize()
        return a, b, c

    before = None
    for k, formulation in enumerate((first, 1 - first, first, first, 1 - first)):
        state = u * (1.0 - 0.1 * k)
        lsmf._check(lsmf._lib.lsmf_set_formulation(op._h, formulation))
        filler = [torch.full((1 << e,), float("nan"), dtype=torch.float64, device=device) for e in range(4, 20)]
        torch.cuda.synchronize()
        if before is not None:
            for a, b in zip(replay(), before):
                assert torch.equal(a, b), (k, "before cache()")
        op.set_linearization(torch.tensor(state, device=device))
        op.cache()
        ref = oracle.OracleOperator(dim, p, mesh.cell_nodes, mesh.coords, np.zeros(mesh.n_dofs, np.uint8),
                                    caching="tensor4", formulation=formulation)
        if nc is not None:
            ref.set_node_constraints(*nc)
        ref.set_material(mu, lam)
        ref.set_linearization(state)
        ref.cache()
        expect = ref.vmult(v)
        for _ in range(2):
            before = replay()
            for a, b in zip(before, eager()):
                assert torch.equal(a, b), (k, formulation)
        assert np.abs(before[0].double().cpu().numpy() - expect).max() < tol * np.abs(expect).max(), (k, formulation)
        del filler


def test_vcycle_follows_the_fine_operator(device):
    """the captured V-cycle runs the caller's finest operator: after a change of
    its formulation it is the eager V-cycle's again, bit by bit"""
    import torch
    rng = np.random.default_rng(2)
    mu, lam = 1.0 + rng.random(512), 2.0 + rng.random(512)
    results = []
    for graph in (1, 0):
        o = lsmf.solver_options(dim=3, degree=2, n_q_1d=3, n_cells_coarse=[2, 2, 2], n_levels=3, caching="tensor4",
                                mg_caching="tensor4", mg_precision="fp64", smoother_degree=3, coarse_solver="direct",
                                use_graph=graph, dirichlet={0: ([0, 1, 2], [0.0] * 3), 1: ([0], [0.01])})
        s = lsmf.Solver(o, mu, lam)
        n = s.n_dofs()
        r = torch.tensor(np.random.default_rng(3).standard_normal(n), device=device)
        z = torch.empty_like(r)
        u = 1e-4 * np.random.default_rng(4).standard_normal(n)
        s.set_state(u)
        s.precondition(z, r)
        out = [z.clone()]
        op = lsmf._lib.lsmf_solver_fine_operator(s._h)
        ud = torch.tensor(u, device=device)
        torch.cuda.synchronize()
        for formulation in (0, 1):
            lsmf._check(lsmf._lib.lsmf_set_formulation(op, formulation))
            lsmf._check(lsmf._lib.lsmf_set_linearization(op, ud.data_ptr(), None))
            lsmf._check(lsmf._lib.lsmf_cache(op, None))
            lsmf._check(lsmf._lib.lsmf_compute_diagonal(op, None))
            for _ in range(3):
                z.fill_(float("nan"))
                torch.cuda.synchronize()
                s.precondition(z, r)
                out.append(z.clone())
        results.append(out)
    for a, b in zip(*results):
        assert torch.equal(a, b)
    assert not torch.equal(results[0][0], results[0][1]) and torch.equal(results[0][0], results[0][-1])


@pytest.mark.parametrize("precision,layout,n", [("fp64", "auto", [36, 40, 36]), ("fp32", "auto", [36, 40, 36]),
                                                ("fp64", "cells", [28, 28, 28])], ids=lambda v: str(v).replace(" ", ""))
def test_replays_of_many_tiles(precision, layout, n, device):
    """more than 256 workgroups per colour, where the formulations' kernels are
    recorded one after the other: replays give the eager products' bits"""
    import torch
    print(f"[recorded] {n} {precision} {layout}", flush=True)
    mesh = lsmf.Mesh(3, 2, n)
    rng = np.random.default_rng(3)
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.02, 7)
    op = lsmf.NeoHookOperator(mesh, precision=precision, caching="tensor4", layout=layout)
    op.set_material(1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells))
    ud = torch.tensor(u, device=device)
    x = torch.tensor(rng.standard_normal(mesh.n_dofs), device=device).to(op.dtype)
    y, z = torch.empty_like(x), torch.empty_like(x)
    op.set_linearization(ud)
    op.cache()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op.vmult(y, x)
    results = []
    for formulation in (1, 0, 1):
        lsmf._check(lsmf._lib.lsmf_set_formulation(op._h, formulation))
        op.set_linearization(ud)
        op.cache()
        for _ in range(2):
            y.fill_(float("nan"))
            graph.replay()
            op.vmult(z, x)
            torch.cuda.synchronize()
            assert torch.equal(y, z), formulation
        results.append(z.clone())
    assert torch.equal(results[0], results[2]) and not torch.equal(results[0], results[1])
