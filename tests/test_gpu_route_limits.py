"""GPU: which path a call takes around the limits of the dispatch rules, from the
launch counts of the library's kernel timers."""
from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _launched(call, kernel):
    import spacecharge as sc
    with sc.KernelTimer() as t:
        call()
    return kernel in t.results()


def _uniform(n, T, k=3):
    g = torch.Generator(device=DEV).manual_seed(n)
    return [torch.rand(n, generator=g, device=DEV, dtype=T) * 1.99 - 0.995 for _ in range(k)]


@pytest.mark.parametrize("T,grid,few,many", [
    (torch.float32, (32, 32, 32), 125_000, 125_001), (torch.float32, (128, 128, 128), 190_000, 340_000),
    (torch.float32, (256, 256, 256), 599_186, 800_000), (torch.float64, (16, 16, 16), 1, 160_001),
    (torch.float64, (100, 100, 100), 166_666, 250_000), (torch.float64, (128, 128, 128), 320_000, 690_000)])
def test_field_copy_of_the_interpolation(T, grid, few, many):
    import spacecharge as sc
    mesh, copied = (sc.Mesh3D(grid, (-1.0,) * 3, (1.0,) * 3, T=T) for _ in range(2))
    mesh.efield.normal_()
    copied.efield.copy_(mesh.efield)
    copied.set_field_layout(1)
    for n in (few, many):
        p = _uniform(n, T)
        assert _launched(lambda: sc.interpolate_field(mesh, *p), "interleave") == (n == many), n
        for a, b in zip(sc.interpolate_field(mesh, *p), sc.interpolate_field(copied, *p)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("T,grid,few,many", [
    (torch.float32, (16, 16, 16), 1_000_000, 17_000_000), (torch.float32, (32, 32, 32), 262_144, 734_000),
    (torch.float32, (48, 48, 48), 77_672, 77_673), (torch.float32, (64, 64, 64), 32_768, 32_769),
    (torch.float64, (32, 32, 32), 524_288, 734_000), (torch.float64, (48, 48, 48), 155_344, 217_482),
    (torch.float64, (64, 64, 64), 57_344, 65_536), (torch.float64, (65, 65, 81), 20_000, 40_000)])
def test_binning_of_the_deposit(T, grid, few, many):
    import spacecharge as sc
    mesh, binned = (sc.Mesh3D(grid, (-1.0,) * 3, (1.0,) * 3, T=T) for _ in range(2))
    binned.set_deposit_tiling(13, 11)
    tiles = 1
    for n in grid:
        tiles *= (n + 14) // 16
    for n in (few, many):
        p = _uniform(n, T, 4)
        # (beyond 64 tiles every count is binned)
        assert _launched(lambda: sc.deposit(mesh, *p), "bin_scatter") == (n == many or tiles > 64), n
        sc.deposit(binned, *p)
        err = float((mesh.rho - binned.rho).double().norm() / binned.rho.double().norm())
        assert err <= (1e-6 if T == torch.float32 else 1e-13)


@pytest.mark.parametrize("T,grid,few,many", [
    (torch.float32, (32, 32, 32), 87_381, 174_762), (torch.float32, (48, 48, 48), 25_890, 25_891),
    (torch.float64, (33, 33, 17), 349_525, 349_526), (torch.float64, (64, 64, 64), 19_114, 21_846)])
def test_binning_of_the_cotangent_deposit(T, grid, few, many):
    import spacecharge as sc
    mesh, binned = (sc.Mesh3D(grid, (-1.0,) * 3, (1.0,) * 3, T=T) for _ in range(2))
    binned.set_deposit_tiling(13, 11)
    for n in (few, many):
        p = _uniform(n, T, 6)
        got = []
        assert _launched(lambda: got.append(sc.interpolate_adjoint(mesh, *p, positions=False)[0]),
                         "bin_scatter") == (n == many), n
        want = sc.interpolate_adjoint(binned, *p, positions=False)[0]
        err = float((got[0] - want).double().norm() / want.double().norm())
        assert err <= (1e-6 if T == torch.float32 else 1e-13)


def _workspace(halves, grid, size):
    """Bytes of the solver's workspace for these transform half-lengths."""
    (hx, hy, hz), (_, _, mz) = halves, grid
    kp = (hx + 1 + 31) // 32 * 32
    spec, gf, gi = mz * 2 * hy * kp, (hz + 1) * (hy + 1) * kp, 2 * hz * (hy + 1) * kp
    fn, rn = (hx + 1) * (hy + 1) * (3 * hz + 1), (hy + 1) * kp * (3 * hz - 1)
    return 8 * size * spec + 3 * size * gf + 6 * size * gi + 24 * fn + 3 * size * rn


# z beyond the register lengths: x and y padded to them only where that is faster
@pytest.mark.parametrize("T,grid,halves", [
    (torch.float64, (51, 51, 300), (54, 54, 300)), (torch.float64, (33, 47, 300), (36, 48, 300)),
    (torch.float64, (33, 51, 600), (35, 54, 600)), (torch.float64, (26, 257, 257), (27, 270, 270)),
    (torch.float64, (257, 26, 26), (270, 32, 32)), (torch.float32, (51, 51, 300), (64, 64, 300)),
    (torch.float32, (51, 51, 600), (54, 54, 600)), (torch.float32, (33, 47, 600), (36, 48, 600))])
def test_padding_of_the_transforms(T, grid, halves):
    import spacecharge as sc
    g = torch.Generator(device=DEV).manual_seed(3)
    rho = torch.rand(grid, generator=g, device=DEV, dtype=T)
    out = []
    for generic in (False, True):
        m = sc.Mesh3D(grid, (-1e-3, -1e-3, 1e-4), (1e-3, 1.2e-3, 2e-3), T=T, gamma=1.5)
        if generic:
            m.force_generic_transforms()
        m.rho.copy_(rho)
        for cath in (False, True):
            sc.solve(m, at_cathode=cath)
            out.append(m.efield.double())
        assert m.workspace_bytes == _workspace(halves, grid, T.itemsize)
        del m
    for a, b in ((out[0], out[2]), (out[1], out[3])):
        for c in range(3):
            d = (a[..., c] - b[..., c]).norm() / b[..., c].norm()
            assert float(d) <= (1e-5 if T == torch.float32 else 1e-12)


def _forks(call):
    """Whether the captured call runs kernels beside each other."""
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    hip = ctypes.CDLL("libamdhip64.so")
    nodes, edges = ctypes.c_size_t(), ctypes.c_size_t()
    g = ctypes.c_void_p(graph.raw_cuda_graph())
    assert hip.hipGraphGetNodes(g, None, ctypes.byref(nodes)) == 0
    assert hip.hipGraphGetEdges(g, None, None, ctypes.byref(edges)) == 0
    return edges.value >= nodes.value  # a chain has one edge fewer than nodes


# a Green build with generic passes beside the deposit, on the caller's stream only
# where it is smaller than one of the register engines
@pytest.mark.parametrize("T,P,grid,beside", [
    (torch.float32, torch.float64, (20, 20, 20), False), (torch.float32, torch.float64, (33, 33, 33), True),
    (torch.float32, torch.float64, (100, 20, 20), True), (torch.float32, torch.float64, (32, 32, 32), False),
    (torch.float32, torch.float64, (50, 64, 32), True), (torch.float32, torch.float64, (32, 32, 50), False),
    (torch.float32, torch.float64, (64, 64, 64), True), (torch.float32, torch.float32, (33, 33, 33), False),
    (torch.float64, torch.float64, (300, 8, 8), False), (torch.float64, torch.float64, (48, 48, 48), True)])
def test_stream_of_the_green_build(T, P, grid, beside):
    import spacecharge as sc
    mesh, big = (sc.Mesh3D(g, (-1.0,) * 3, (1.0,) * 3, T=T) for g in (grid, (64, 64, 64)))
    p = _uniform(3000, P, 4)
    for m in (big, mesh):  # the larger one makes the library's second stream

        def step(m=m):
            p[3].mul_(1.0)  # one first node of the graph
            sc.deposit(m, *p)
            sc.solve(m)
        step()
    torch.cuda.synchronize()
    assert _forks(step) == beside


# lengths along z at which the generic kernel is the faster one
@pytest.mark.parametrize("kind,T,n", [
    ("field", torch.float64, 40), ("field", torch.float64, 80), ("adjoint", torch.float64, 40),
    ("adjoint", torch.float64, 96), ("adjoint", torch.float64, 192), ("adjoint", torch.float32, 40),
    ("adjoint", torch.float32, 160), ("adjoint", torch.float32, 200)])
def test_cathode_convolution_is_no_slower_than_the_generic_one(kind, T, n):
    import spacecharge as sc
    grid = (128, 128, n)
    g = torch.rand((*grid, 3), device=DEV, dtype=T)
    best, out = [], []
    for generic in (False, True):
        m = sc.Mesh3D(grid, (-1e-3, -1e-3, 1e-4), (1e-3, 1.2e-3, 2e-3), T=T, gamma=1.5)
        m.force_generic_transforms(generic)
        m.rho.copy_(g[..., 0])

        def call():
            if kind == "adjoint":
                return sc.solve_adjoint(m, g, at_cathode=True)
            sc.solve(m, at_cathode=True)
            return m.efield
        out.append(call().double())
        times = []
        for _ in range(5):
            with sc.KernelTimer() as t:
                for _ in range(4):
                    call()
            times.append(t.results()["zconv"][0])
        best.append(min(times))
    print(f"{kind} {T} {n}: {best[0]:.3f} ms, generic {best[1]:.3f}", flush=True)
    assert float((out[0] - out[1]).norm() / out[1].norm()) <= (1e-5 if T == torch.float32 else 1e-12)
    assert best[0] <= 1.15 * best[1]
