"""GPU: the x and y passes in one kernel (short or equal x and y axes), against the
generic engine's separate passes on the same Green spectra.

Both engines' transforms err by about eps per butterfly level, at most 21 levels
(the padded volume is below 2^21 per transform) forward and backward: 42 eps each,
relative L2 84 eps between the two; 2e-14 and 1e-5 allow twice that."""
from __future__ import annotations

import pytest
import torch

from _common import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _meshes(grid, T, n=2):
    import spacecharge as sc
    out = []
    for k in range(n):
        m = sc.Mesh3D(grid, (-1e-2, -2e-2, 1e-3), (1e-2, 1e-2, 3e-2), T=T, gamma=2.0)
        g = torch.Generator(device=DEV).manual_seed(5 + k)
        m.rho.copy_(torch.rand(m.rho.shape, generator=g, device=DEV, dtype=torch.float64).to(T))
        out.append(m)
    return sc, out


# pairs of short lengths with padded and exact axes, one plane, each longer equal pair
# (the last ones take the plane in Float32 only), and a pair just beyond
@pytest.mark.parametrize("T", [torch.float32, torch.float64])
@pytest.mark.parametrize("grid", [(2, 2, 2), (8, 12, 2), (5, 24, 9), (16, 31, 8), (32, 9, 16),
                                  (23, 32, 40), (36, 33, 6), (37, 40, 12), (47, 41, 9), (50, 49, 16),
                                  (64, 61, 10), (65, 72, 8), (73, 80, 7), (32, 33, 8)])
def test_plane_equals_separate_passes(grid, T):
    sc, (m, _) = _meshes(grid, T)
    m.set_green_reuse(True)  # both engines on one set of Green spectra
    tol = 1e-5 if T == torch.float32 else 2e-14
    g = torch.randn(m.efield.shape, generator=torch.Generator(device=DEV).manual_seed(9), device=DEV,
                    dtype=torch.float64).to(T)

    def run(what):
        if what == "potential":
            return sc.solve_potential(m).clone()
        if what.startswith("adjoint"):
            return sc.solve_adjoint(m, g, at_cathode=what.endswith("cathode")).clone()
        sc.solve(m, at_cathode=what == "cathode")
        return m.efield.clone()

    for what in ("field", "adjoint", "cathode", "adjoint cathode", "potential"):
        m.force_generic_transforms(False)
        res = [run(what)]
        m.force_generic_transforms()
        res.append(run(what))
        err = rel_l2(res[0].double().cpu().numpy(), res[1].double().cpu().numpy())
        print(f"plane {grid} {T} {what}: {err:.2e}")
        assert err <= tol


@pytest.mark.parametrize("T", [torch.float32, torch.float64])
@pytest.mark.parametrize("grid", [(16, 31, 8), (50, 49, 16)])
def test_batched_plane_equals_single(grid, T):
    sc, ms = _meshes(grid, T, 3)
    want = []
    for m in ms:
        sc.solve(m)
        want.append(m.efield.clone())
        m.efield.zero_()
    sc.solve_batched(ms)
    torch.cuda.synchronize()
    for m, w in zip(ms, want):
        assert torch.equal(m.efield, w)
