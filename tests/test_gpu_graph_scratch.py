"""GPU: one eager call reserves the scratch of every later call of at most as many
particles, by whichever path it runs, so that a captured step stays valid after
eager calls that take another path, and nothing is allocated inside a capture.

Float32 meshes: equal to the bits of the same call on a mesh that is never captured.
Float64 ones add in an order that varies: 1e-13, the suite's gate for the deposit."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from _common import gaussian, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _bunch(n, seed, dtype):
    x, y, z = gaussian(n, (1e-3, 1e-3, 2e-3), seed)
    return [torch.as_tensor(a, dtype=dtype, device=DEV) for a in (x, y, z, np.full(n, 1e-9 / n))]


def _capture(fn):
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _same(a, b):
    if a.dtype == torch.float32:
        return torch.equal(a, b)
    return rel_l2(a.cpu().numpy(), b.cpu().numpy()) <= 1e-13


# many: binned; few: without binning
@pytest.mark.parametrize("T,many,few", [(torch.float32, 500_000, 200_000), (torch.float64, 600_000, 500_000)])
@pytest.mark.parametrize("captured", ["many", "few"])
def test_captured_deposit_and_an_eager_one_of_another_size(T, many, few, captured):
    import spacecharge as sc
    grid = (32, 32, 32)
    big = _bunch(many, 3, T)
    small = [a[:few].clone() for a in big]
    mesh, ref = (sc.Mesh3D(grid, *big[:3], T=T) for _ in range(2))
    sc.deposit(mesh, *big)
    parts, other = (big, small) if captured == "many" else (small, big)
    graph, _ = _capture(lambda: sc.deposit(mesh, *parts))
    for rep in range(3):
        print(f"{captured} {T} {rep}", flush=True)
        if captured == "few" or rep:
            sc.deposit(mesh, *other)
            sc.deposit(ref, *other)
            assert _same(mesh.rho, ref.rho)
        parts[3].mul_(1.25)
        graph.replay()
        sc.deposit(ref, *parts)
        torch.cuda.synchronize()
        assert _same(mesh.rho, ref.rho), rep


@pytest.mark.parametrize("T", [torch.float32, torch.float64])
@pytest.mark.parametrize("captured", ["batched", "single"])
def test_captured_batched_deposit_and_single_ones(T, captured):
    import spacecharge as sc
    specs = [((16, 16, 16), 10_000), ((32, 32, 32), 100_000), ((64, 64, 64), 30_000)]
    parts = [_bunch(n, 40 + n, T) for _, n in specs]
    meshes, refs = ([sc.Mesh3D(g, *p[:3], T=T) for (g, _), p in zip(specs, parts)] for _ in range(2))

    def batched(ms):
        sc.deposit_batched(ms, *[[p[k] for p in parts] for k in range(4)])

    def single(ms):
        for m, p in zip(ms, parts):
            sc.deposit(m, *p)

    inside, outside = (batched, single) if captured == "batched" else (single, batched)
    if captured == "batched":
        batched(refs)  # the context's descriptor table
    outside(meshes)  # the only eager call before the capture takes the other path
    graph, _ = _capture(lambda: inside(meshes))
    for rep in range(3):
        print(f"{captured} {T} {rep}", flush=True)
        for p in parts:
            p[3].mul_(1.25)
        outside(meshes)
        graph.replay()
        inside(refs)
        torch.cuda.synchronize()
        for m, r in zip(meshes, refs):
            assert _same(m.rho, r.rho), rep


@pytest.mark.parametrize("T", [torch.float32, torch.float64])
def test_captured_cotangent_deposit_with_a_tiling_set_after_the_eager_one(T):
    """Three channels: eager without binning, captured binned (a tiling of the mesh's own)."""
    import spacecharge as sc
    grid, n = (32, 32, 32), 50_000
    x, y, z, q = _bunch(n, 9, T)
    g = [torch.randn_like(x) for _ in range(3)]
    mesh, ref = (sc.Mesh3D(grid, x, y, z, T=T) for _ in range(2))
    want = sc.interpolate_adjoint(mesh, x, y, z, *g)[0]
    for m in (mesh, ref):
        m.set_deposit_tiling(14, 12)  # no more chunks than the default's
    out = torch.empty_like(want)
    graph, _ = _capture(lambda: out.copy_(sc.interpolate_adjoint(mesh, x, y, z, *g)[0]))
    for rep in range(2):
        graph.replay()
        got = sc.interpolate_adjoint(ref, x, y, z, *g)[0]
        torch.cuda.synchronize()
        assert _same(out, got)
        for c in g:
            c.mul_(0.5)


# few: gathered without the field copy
@pytest.mark.parametrize("T", [torch.float32, torch.float64])
@pytest.mark.parametrize("call", ["single", "batched", "adjoint"])
def test_captured_interpolation_after_an_eager_one_of_few_particles(T, call):
    import spacecharge as sc
    many = _bunch(300_000, 5, T)[:3]
    few = [a[:1000].clone() for a in many]
    mesh, ref = (sc.Mesh3D((32, 32, 32), *many, T=T) for _ in range(2))
    g = torch.Generator(device=DEV).manual_seed(2)
    ef = torch.randn(mesh.efield.shape, generator=g, device=DEV, dtype=T)
    cot = [torch.randn(many[0].shape, generator=g, device=DEV, dtype=T) for _ in range(3)]

    def run(m, p):
        if call == "batched":
            return sc.interpolate_batched([m], *[[a] for a in p])[0]
        if call == "adjoint" and len(p[0]) > 1000:
            return sc.interpolate_adjoint(m, *p, *cot)[1:]
        return sc.interpolate_field(m, *p)

    if call == "adjoint":  # its deposit's scratch
        sc.interpolate_adjoint(mesh, *many, *cot, positions=False)
    for m in (mesh, ref):
        m.efield.copy_(ef)
    run(mesh, few)
    graph, out = _capture(lambda: run(mesh, many))
    for rep in range(2):
        graph.replay()
        want = run(ref, many)
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a, b)
        for m in (mesh, ref):
            m.efield.mul_(0.5)
