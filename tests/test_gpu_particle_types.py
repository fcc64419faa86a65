"""GPU: a solve's bits follow from what it solves, not from what ran on the mesh or
beside it before.  Float32 meshes take other transform lengths and kernels where
their charges were deposited from Float64 particles; neither an earlier deposit or
solve of the other kind nor the other meshes of a batch may show in the result."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
GRIDS = [(20, 33, 26), (32, 32, 32), (50, 12, 9)]  # padded, powers of two, padded either way


def _bunch(T, seed=5, n=4000):
    g = torch.Generator(device=DEV).manual_seed(seed)
    p = [torch.rand(n, generator=g, device=DEV, dtype=torch.float64) for _ in range(4)]
    return [a.to(T) for a in p]


def _mesh(grid):
    import spacecharge as sc
    return sc.Mesh3D(grid, (0.0,) * 3, (1.0,) * 3, T=torch.float32, gamma=2.0)


def _step(mesh, p, kind="field"):
    import spacecharge as sc
    sc.deposit(mesh, *p)
    if kind == "potential":
        return sc.solve_potential(mesh).clone()
    sc.solve(mesh, at_cathode=kind == "cathode")
    return torch.stack(sc.interpolate_field(mesh, *p[:3]))


@pytest.mark.parametrize("kind", ["field", "cathode", "potential"])
@pytest.mark.parametrize("reuse", [False, True])
@pytest.mark.parametrize("grid", GRIDS)
def test_result_does_not_depend_on_earlier_particle_types(grid, reuse, kind):
    narrow, wide = _bunch(torch.float32), _bunch(torch.float64, 6)
    want = {}
    for p in (narrow, wide):
        want[p[0].dtype] = _step(_mesh(grid), p, kind)
    mesh = _mesh(grid)
    mesh.set_green_reuse(reuse)
    for p in (narrow, wide, wide, narrow, wide, narrow):
        assert torch.equal(_step(mesh, p, kind), want[p[0].dtype]), p[0].dtype


@pytest.mark.parametrize("grid", GRIDS)
def test_added_and_cleared_charges(grid):
    import spacecharge as sc
    narrow, wide = _bunch(torch.float32), _bunch(torch.float64, 6)
    want_wide, want_narrow = _step(_mesh(grid), wide), _step(_mesh(grid), narrow)
    zero = [*narrow[:3], torch.zeros_like(narrow[3])]
    mesh = _mesh(grid)
    _step(mesh, narrow)
    sc.deposit(mesh, *wide)
    sc.deposit(mesh, *zero, clear=False)  # rho still holds the Float64 particles' charges
    sc.solve(mesh)
    assert torch.equal(torch.stack(sc.interpolate_field(mesh, *wide[:3])), want_wide)
    sc.clear_mesh(mesh)
    sc.deposit(mesh, *narrow, clear=False)
    sc.solve(mesh)
    assert torch.equal(torch.stack(sc.interpolate_field(mesh, *narrow[:3])), want_narrow)


@pytest.mark.parametrize("grid", GRIDS)
def test_adjoint_does_not_depend_on_earlier_particle_types(grid):
    import spacecharge as sc

    def grad(mesh, p):
        g = sc.interpolate_adjoint(mesh, *p[:3], *p[1:4], positions=False)[0]
        return sc.solve_adjoint(mesh, g).clone()

    narrow, wide = _bunch(torch.float32), _bunch(torch.float64, 6)
    want = {p[0].dtype: grad(_mesh(grid), p) for p in (narrow, wide)}
    mesh = _mesh(grid)
    for p in (wide, narrow, narrow, wide):
        _step(mesh, p)
        for q in (narrow, wide):
            assert torch.equal(grad(mesh, q), want[q[0].dtype])


@pytest.mark.parametrize("grid", GRIDS)
def test_adjoint_of_given_cotangents_follows_the_charges(grid):
    """Without a cotangent deposit the adjoint takes the field solve's lengths, and its
    Green spectra where they are reused."""
    import spacecharge as sc
    narrow, wide = _bunch(torch.float32), _bunch(torch.float64, 6)
    g = torch.rand((*grid, 3), generator=torch.Generator(device=DEV).manual_seed(1), device=DEV)
    mesh = _mesh(grid)
    mesh.set_green_reuse()
    for p in (narrow, wide, narrow):
        fresh = _mesh(grid)
        sc.deposit(fresh, *p)
        want = sc.solve_adjoint(fresh, g).clone()
        sc.interpolate_adjoint(mesh, *wide[:3], *wide[1:4], positions=False)
        sc.deposit(mesh, *p)
        sc.solve(mesh)
        with sc.KernelTimer() as t:
            got = sc.solve_adjoint(mesh, g)
        assert not any(k.startswith("green") for k in t.results())
        assert torch.equal(got, want)


@pytest.mark.parametrize("order", [(0, 1, 0, 1), (1, 0, 1, 0)])
@pytest.mark.parametrize("grid", [(32, 32, 32), (16, 16, 16), (20, 33, 26)])
def test_batch_of_both_kinds_equals_single_solves(grid, order):
    import spacecharge as sc
    parts = [_bunch((torch.float32, torch.float64)[k], 20 + i) for i, k in enumerate(order)]
    want = []
    for p in parts:
        m = _mesh(grid)
        sc.deposit(m, *p)
        sc.solve(m)
        want.append(m.efield.clone())
    meshes = [_mesh(grid) for _ in parts]
    for rep in range(2):
        for m, p in zip(meshes, parts):
            sc.deposit(m, *p)
        sc.solve_batched(meshes)
        torch.cuda.synchronize()
        for m, w in zip(meshes, want):
            assert torch.equal(m.efield, w)
            m.efield.zero_()


def test_captured_step_of_either_kind_after_one_of_the_other():
    """One eager step of either kind prepares the capture of the other."""
    grid = (20, 33, 26)
    narrow, wide = _bunch(torch.float32), _bunch(torch.float64, 6)
    for first, second in ((narrow, wide), (wide, narrow)):
        want = _step(_mesh(grid), second)
        mesh = _mesh(grid)
        _step(mesh, first)
        _step(_mesh(grid), second)
        import spacecharge as sc
        sc.sort_permutation(mesh, *second[:3])  # records of the wider type
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = _step(mesh, second)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)
            _step(mesh, first)
