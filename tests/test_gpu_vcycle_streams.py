"""The V-cycle against its definition and beside other work.

The smoother's vector updates run inside the products' launches, in a buffer of
the operator that belongs to the solver's stream.  A V-cycle put together here
from separate operators' products, the solver's transfers and torch's vector
updates has to give the same result; and one graph, replayed many times while
the finest operator's products run on other streams, the same bits.

Tolerance of the first: a product's relative error is about 1e-15 of its largest
entry, a V-cycle chains 2 (degree + 1) of them per level and amplifies none
(the Chebyshev polynomials are bounded by 1 on the spectrum), and the inverse
of the coarse matrix loses its condition number, about 1e3: 1e-11 of the
largest entry.
"""
import ctypes

import numpy as np
import pytest

import lsmf

pytestmark = pytest.mark.gpu


def solver(p, coarse, levels, degree, graph, mu, lam):
    o = lsmf.solver_options(dim=3, degree=p, n_q_1d=p + 1, n_cells_coarse=coarse, n_levels=levels, caching="tensor4",
                            mg_caching="tensor4", mg_precision="fp64", smoother_degree=degree, coarse_solver="direct",
                            use_graph=graph, dirichlet={0: ([0, 1, 2], [0.0] * 3), 1: ([0], [0.01])})
    n = int(np.prod(coarse)) * 8 ** (levels - 1)
    return o, lsmf.Solver(o, np.full(n, mu), np.full(n, lam))


@pytest.mark.parametrize("p,coarse,levels", [(2, [1, 1, 1], 3), (2, [3, 1, 2], 2), (4, [1, 1, 1], 2), (1, [2, 2, 2], 3)],
                         ids=lambda v: str(v).replace(" ", ""))
def test_vcycle_is_products_transfers_and_updates(p, coarse, levels, device):
    import torch
    print(f"[vcycle] p={p} {coarse} {levels}", flush=True)
    mu, lam, degree = 1.3, 2.1, 4
    o, s = solver(p, coarse, levels, degree, 1, mu, lam)
    n = s.n_dofs()
    rng = np.random.default_rng(4)
    mesh = lsmf.Mesh(3, p, [c << (levels - 1) for c in coarse])
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.01, 3)
    s.set_state(u)
    ops, cons, states = [None] * levels, [None] * levels, [None] * levels
    states[-1] = torch.tensor(u, device=device)
    for l in range(levels - 1, -1, -1):
        m = lsmf.Mesh(3, p, [c << l for c in coarse])
        if l < levels - 1:
            states[l] = torch.empty(m.n_dofs, dtype=torch.float64, device=device)
            s.transfer(l + 1, 2, states[l], states[l + 1])
        mask = m.constrained_mask({0: [0, 1, 2], 1: [0]})
        cons[l] = torch.tensor(mask, device=device).bool()
        ops[l] = lsmf.NeoHookOperator(m, caching="tensor4", constrained=mask)
        ops[l].set_material(np.full(m.n_cells, mu), np.full(m.n_cells, lam))
        ops[l].set_linearization(states[l])
        ops[l].cache()
        ops[l].compute_diagonal()

    def product(l, x):
        y = torch.empty_like(x)
        ops[l].vmult(y, x)
        return y

    def chebyshev(l, x, b):
        lmax = 1.2 * s.level_info(l)[0]
        alpha = lmax / o.smoothing_range
        theta, delta = 0.5 * (lmax + alpha), 0.5 * (lmax - alpha)
        invd = ops[l].inverse_diagonal()
        d = invd * (b if x is None else b - product(l, x)) / theta
        x = d.clone() if x is None else x + d
        rho, sigma = delta / theta, theta / delta
        for _ in range(degree - 1):
            new = 1.0 / (2.0 * sigma - rho)
            d = new * rho * d + 2.0 * new / delta * invd * (b - product(l, x))
            rho = new
            x = x + d
        return x

    eye = torch.eye(ops[0].m(), dtype=torch.float64, device=device)
    A0 = torch.empty_like(eye)
    ops[0].vmult_batched(A0, eye)

    def vcycle(l, b):
        if l == 0:
            return torch.tensor(np.linalg.solve(A0.cpu().numpy(), b.cpu().numpy()), device=device)
        x = chebyshev(l, None, b)
        coarse_b = torch.empty(ops[l - 1].m(), dtype=torch.float64, device=device)
        s.transfer(l, 1, coarse_b, b - product(l, x))
        coarse_b[cons[l - 1]] = 0
        up = torch.empty_like(b)
        s.transfer(l, 0, up, vcycle(l - 1, coarse_b))
        x = x + up
        x[cons[l]] = 0
        return chebyshev(l, x, b)

    r = torch.tensor(rng.standard_normal(n), device=device)
    z = torch.empty_like(r)
    torch.cuda.synchronize()
    s.precondition(z, r)
    expect = vcycle(levels - 1, r)
    assert float((z - expect).abs().max()) < 1e-11 * float(expect.abs().max())


@pytest.mark.parametrize("p,coarse,levels", [(2, [2, 2, 2], 3), (4, [1, 1, 1], 3)], ids=lambda v: str(v).replace(" ", ""))
def test_replays_beside_products_on_other_streams(p, coarse, levels, device):
    import torch
    print(f"[replay] p={p} {coarse} {levels}", flush=True)
    results = []
    for graph in (1, 0):
        _, s = solver(p, coarse, levels, 4, graph, 1.3, 2.1)
        n = s.n_dofs()
        s.set_state(1e-5 * np.random.default_rng(4).standard_normal(n))
        fine = lsmf._lib.lsmf_solver_fine_operator(s._h)
        rng = np.random.default_rng(5)
        r = torch.tensor(rng.standard_normal(n), device=device)
        xs = [torch.tensor(rng.standard_normal(n), device=device) for _ in range(2)]
        ys = [torch.empty_like(r) for _ in range(2)]
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        torch.cuda.synchronize()

        def products(k):
            for x, y, st in zip(xs, ys, streams):
                lsmf._check(lsmf._lib.lsmf_vmult(fine, y.data_ptr(), x.data_ptr(), 0, lsmf.MASK["default"],
                                                 ctypes.c_void_p(st.cuda_stream)))

        products(0)
        torch.cuda.synchronize()
        expect = [y.clone() for y in ys]
        z = torch.empty_like(r)  # one z and r throughout: one graph
        first = None
        for k in range(6):
            z.fill_(float("nan"))
            for y in ys:
                y.fill_(float("nan"))
            torch.cuda.synchronize()
            for _ in range(20):
                products(k)
            s.precondition(z, r)
            products(k)
            torch.cuda.synchronize()
            if first is None:
                first = z.clone()
                assert bool(torch.isfinite(first).all())
            assert torch.equal(z, first), k
            assert torch.equal(ys[0], expect[0]) and torch.equal(ys[1], expect[1]), k
        results.append(first)
    assert torch.equal(results[0], results[1])
