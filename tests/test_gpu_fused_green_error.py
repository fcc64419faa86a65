"""GPU: the Green function built in one kernel (small meshes) is as close to a plain
64-bit evaluation as that of the separate kernels (the generic engine's).

Both round the same terms, so their errors should agree.  The transforms differ and
add their own rounding in squares: at most a few 1e-16 (see test_gpu_plane.py)
against 8e-15 and more on these meshes, 0.4% of the error: gated at 1%."""
from __future__ import annotations

import os
import sys

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


@pytest.mark.parametrize("grid", [(24, 24, 24), (20, 28, 36), (32, 32, 32), (36, 36, 36)])
def test_error_against_64_bits(grid):
    import spacecharge as sc
    from perf.cases import _convolve
    err = {False: 0.0, True: 0.0}
    for k in range(10):
        g = torch.Generator(device=DEV).manual_seed(k)
        rho = torch.rand(grid, generator=g, device=DEV, dtype=torch.float64) * 1e-12
        for generic in (False, True):
            m = sc.Mesh3D(grid, (-1e-3, -1.1e-3, -2e-3), (1e-3, 1.2e-3, 2e-3), T=torch.float64,
                          gamma=(1.0, 1.0, 3.0)[k % 3])
            m.force_generic_transforms(generic)
            m.rho.copy_(rho)
            sc.solve(m)
            if not generic:
                ex = _convolve(rho.permute(2, 1, 0).contiguous(), (0, 1, 2), grid, m.min_bounds,
                               m.max_bounds, m.delta, m.gamma, False)
                ex = torch.stack(ex, -1).permute(2, 1, 0, 3)
            err[generic] += float((m.efield - ex).norm() / ex.norm())
    print(f"fused Green build {grid}: {err[False] / 10:.4e}, separate {err[True] / 10:.4e}")
    assert err[False] <= 1.01 * err[True]
