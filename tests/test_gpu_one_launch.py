"""Products in one launch over all tiles (the operator's first stream) against
the coloured launches (any other stream, captured calls, batched products):
the same sums in the same order, so the same bits, for set, add, plain and
phase-masked products, the diagonal, the residual and its VJP, at meshes of one cell, less
than one tile, ragged and several tiles per direction.
"""
import threading

import numpy as np
import pytest

import lsmf

pytestmark = pytest.mark.gpu

MESHES = [(2, 1, [1, 1]), (2, 2, [9, 13]), (2, 4, [11, 5]), (3, 1, [9, 5, 5]), (3, 2, [1, 1, 1]), (3, 2, [19, 5, 3]),
          (3, 2, [9, 4, 2]), (3, 4, [9, 3, 2]), (3, 4, [4, 1, 1])]


def operator(dim, p, n, caching, precision, device):
    import torch
    mesh = lsmf.Mesh(dim, p, n)
    rng = np.random.default_rng(5)
    op = lsmf.NeoHookOperator(mesh, precision=precision, caching=caching,
                              constrained=mesh.constrained_mask({0: list(range(dim)), 1: [0]}))
    op.set_material(1.0 + rng.random(mesh.n_cells), 2.0 + rng.random(mesh.n_cells))
    u, _ = lsmf.smooth_displacement(mesh.coords, 0.02, 3)
    op.set_linearization(torch.tensor(u, device=device))
    op.cache()
    x = torch.tensor(rng.standard_normal(mesh.n_dofs), device=device).to(op.dtype)
    return op, x


@pytest.mark.parametrize("caching,precision", [("tensor4", "fp64"), ("tensor2", "fp32"), ("scalar", "fp64")])
@pytest.mark.parametrize("dim,p,n", MESHES, ids=lambda v: str(v).replace(" ", ""))
def test_same_bits_as_coloured_launches(dim, p, n, caching, precision, device):
    import torch
    print(f"[one launch] dim={dim} p={p} n={n} {caching} {precision}", flush=True)
    op, x = operator(dim, p, n, caching, precision, device)
    start = torch.linspace(-1, 1, x.numel(), device=device, dtype=op.dtype)

    def all_results(stream):
        out = []
        for kw in ({}, {"mask": "plain"}, {"mask": 0x7 | 0x8}, {"add": True}, {"add": True, "mask": "plain"}):
            y = start.clone() if kw.get("add") else torch.full_like(x, float("nan"))
            op.vmult(y, x, stream=stream, **kw)
            out.append(y)
        op.compute_diagonal(stream=stream)
        out.append(op.diagonal())
        if precision == "fp64":
            r, du = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
            dmu = torch.empty(op.n_cells, dtype=x.dtype, device=device)
            dlam = torch.empty_like(dmu)
            op.residual(r, stream=stream)
            op.residual_vjp(x, du, dmu, dlam, stream=stream)
            out += [r, du, dmu, dlam]
        return out

    first = all_results(None)  # claims the tile buffer
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    with torch.cuda.stream(other):
        second = all_results(other.cuda_stream)
    torch.cuda.synchronize()
    for k, (a, b) in enumerate(zip(first, second)):
        assert torch.equal(a, b), k
    batch = torch.full((2, x.numel()), float("nan"), device=device, dtype=op.dtype)
    op.vmult_batched(batch, torch.stack([x, x]))
    assert torch.equal(batch[0], first[0]) and torch.equal(batch[1], first[0])


def test_streams_threads_and_capture(device):
    """two streams at once, four threads on one stream, and a captured product
    replayed between eager ones give the first product's bits"""
    import torch
    op, x = operator(3, 2, [19, 7, 5], "tensor4", "fp64", device)
    xs = [x * (k + 1.0) for k in range(4)]
    expect = []
    for v in xs:
        y = torch.empty_like(x)
        op.vmult(y, v)
        expect.append(y)
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    ys = [torch.full_like(x, float("nan")) for _ in range(8)]
    torch.cuda.synchronize()
    for k in range(4):
        op.vmult(ys[2 * k], xs[k])
        op.vmult(ys[2 * k + 1], xs[k], stream=other.cuda_stream)
    torch.cuda.synchronize()
    for k in range(4):
        assert torch.equal(ys[2 * k], expect[k]) and torch.equal(ys[2 * k + 1], expect[k])

    stream = torch.cuda.current_stream().cuda_stream
    bad = []

    def work(k):
        out = torch.full_like(x, float("nan"))
        for _ in range(10):
            op.vmult(out, xs[k], stream=stream)
        torch.cuda.synchronize()
        if not torch.equal(out, expect[k]):
            bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad

    graph, y, z = torch.cuda.CUDAGraph(), torch.empty_like(x), torch.empty_like(x)
    with torch.cuda.graph(graph):
        op.vmult(y, x)
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        op.vmult(z, xs[1])
        torch.cuda.synchronize()
        assert torch.equal(y, expect[0]) and torch.equal(z, expect[1])
