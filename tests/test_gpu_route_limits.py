"""GPU: which path a call takes around the limits of the dispatch rules, from the
launch counts of the library's kernel timers.  Particles that fill the mesh measured
slower on the path for few particles from a little beyond the limits on."""
from __future__ import annotations

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
    (torch.float32, (32, 32, 32), 100_000, 100_001), (torch.float32, (128, 128, 128), 100_000, 340_000),
    (torch.float32, (256, 256, 256), 349_525, 800_000), (torch.float64, (16, 16, 16), 1, 100_001),
    (torch.float64, (100, 100, 100), 100_000, 250_000), (torch.float64, (128, 128, 128), 87_381, 690_000)])
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
