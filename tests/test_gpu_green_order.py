"""GPU: the Green-function build on the side stream never overtakes a solve that
still reads the spectra.

The build overwrites the mesh's spectra on a second stream.  It forks where the
step's deposit started, and where no deposit came since the last solve, at the
end of the caller's stream.  Every solve of a sequence must give the bits of the
same solve alone on a fresh mesh, whose build has nothing to overtake.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from _common import gaussian

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GRID = (64, 48, 64)  # spectra beyond the size that is built on the caller's stream
N = 200_000


def _setup(T, reuse=False):
    import spacecharge as sc
    x, y, z = gaussian(N, (1e-3, 1e-3, 2e-3), 21)
    p = [torch.as_tensor(a, dtype=T, device=DEV) for a in (x, y, z + 0.02, np.full(N, 1e-15))]
    mesh = sc.Mesh3D(GRID, *p[:3], T=T)
    if reuse:
        mesh.set_green_reuse(True)
    return sc, mesh, p


def _run(sc, mesh, kind, gamma):
    mesh.gamma = gamma
    if kind == "potential":
        return sc.solve_potential(mesh).clone()
    sc.solve(mesh, at_cathode=kind == "cathode")
    return mesh.efield.clone()


SEQUENCE = [("field", 1.0), ("field", 3.0), ("potential", 1.0), ("cathode", 2.0), ("field", 2.0),
            ("field", 2.0), ("potential", 4.0), ("field", 1.0)]


# deposits: a deposit before each solve, before the first only, or on another
# stream than the solves
@pytest.mark.parametrize("deposits", ["each", "first", "stream"])
@pytest.mark.parametrize("T,reuse", [(torch.float32, False), (torch.float32, True),
                                     (torch.float64, False)])
def test_sequence_of_solves_equals_each_alone(T, reuse, deposits):
    sc, mesh, p = _setup(T, reuse)
    sc.deposit(mesh, *p)
    torch.cuda.synchronize()
    rho = mesh.rho.clone()
    want = []
    for kind, gamma in SEQUENCE:
        _, alone, _ = _setup(T)
        alone.rho.copy_(rho)
        want.append(_run(sc, alone, kind, gamma))
    torch.cuda.synchronize()
    other = torch.cuda.Stream()
    got = []
    for _ in range(3):
        for kind, gamma in SEQUENCE:
            if deposits == "each":
                sc.deposit(mesh, *p)
            elif deposits == "stream":
                other.wait_stream(torch.cuda.current_stream())
                with torch.cuda.stream(other):
                    sc.deposit(mesh, *p)
                torch.cuda.current_stream().wait_stream(other)
            mesh.rho.copy_(rho)  # Float64 deposits differ in the last bits
            got.append(_run(sc, mesh, kind, gamma))
    torch.cuda.synchronize()
    for i, g in enumerate(got):
        assert torch.equal(g, want[i % len(SEQUENCE)]), (i, SEQUENCE[i % len(SEQUENCE)])


# The next two read or write the spectra or the geometry beside the kernels that use
# them if the build forks at the deposit.


@pytest.mark.parametrize("T", [torch.float32, torch.float64])
def test_bounds_between_deposit_and_solve(T):
    """Device-resident bounds computed after the deposit are those that the solve uses."""
    sc, mesh, p = _setup(T)
    sc.deposit(mesh, *p)
    torch.cuda.synchronize()
    rho = mesh.rho.clone()
    want, got = [], []
    for rep in range(4):
        x, y, z = (a * (1.0 + 0.25 * rep) for a in p[:3])
        _, alone, _ = _setup(T)
        alone.update_bounds(x, y, z)
        alone.rho.copy_(rho)
        torch.cuda.synchronize()
        want.append(_run(sc, alone, "cathode" if rep % 2 else "field", 2.0))
        torch.cuda.synchronize()
    for rep in range(4):
        x, y, z = (a * (1.0 + 0.25 * rep) for a in p[:3])
        sc.deposit(mesh, *p)
        mesh.update_bounds(x, y, z)
        mesh.rho.copy_(rho)
        got.append(_run(sc, mesh, "cathode" if rep % 2 else "field", 2.0))
    torch.cuda.synchronize()
    for rep in range(4):
        assert torch.equal(got[rep], want[rep]), rep


@pytest.mark.parametrize("T", [torch.float32, torch.float64])
@pytest.mark.parametrize("batched", [False, True])
def test_replay_between_deposit_and_solve(T, batched):
    """A captured step replayed between an eager deposit and its solve."""
    sc, mesh, p = _setup(T)
    other = _setup(T)[1]

    def captured():
        mesh.gamma = 3.0
        sc.deposit(mesh, *p)
        mesh.rho.copy_(rho)
        if batched:
            sc.solve_batched([mesh, other])
        else:
            sc.solve(mesh)
        return mesh.efield.clone()

    sc.deposit(mesh, *p)
    torch.cuda.synchronize()
    rho = mesh.rho.clone()
    other.rho.copy_(rho)
    want = []
    for gamma in (3.0, 1.0):
        _, alone, _ = _setup(T)
        alone.rho.copy_(rho)
        want.append(_run(sc, alone, "field", gamma))
    for _ in range(2):
        captured()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = captured()
    for rep in range(4):
        sc.deposit(mesh, *p)
        graph.replay()
        mesh.rho.copy_(rho)
        got = _run(sc, mesh, "field", 1.0)
        torch.cuda.synchronize()
        assert torch.equal(out, want[0]), rep
        assert torch.equal(got, want[1]), rep


@pytest.mark.parametrize("T", [torch.float32, torch.float64])
def test_replayed_bounds_between_deposit_and_solve(T):
    """The same with bounds that a graph computes."""
    sc, mesh, p = _setup(T)
    live = [a.clone() for a in p[:3]]
    mesh.update_bounds(*live)
    sc.deposit(mesh, *p)
    _run(sc, mesh, "field", 2.0)
    torch.cuda.synchronize()
    rho = mesh.rho.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        mesh.update_bounds(*live)
    for rep in range(4):
        for a, b in zip(live, p):
            a.copy_(b * (1.0 + 0.25 * rep))
        _, alone, _ = _setup(T)
        alone.update_bounds(*live)
        alone.rho.copy_(rho)
        want = _run(sc, alone, "field", 2.0)
        torch.cuda.synchronize()
        sc.deposit(mesh, *p)
        graph.replay()
        mesh.rho.copy_(rho)
        got = _run(sc, mesh, "field", 2.0)
        torch.cuda.synchronize()
        assert torch.equal(got, want), rep
