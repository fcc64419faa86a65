"""The interpolation without the interleaved field copy, and where the rule
switches: the same bits as with the copy (layout 1) for every type pair,
including clamped and non-finite coordinates, device bounds and the last nodes
of every axis."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("pt,mt", [(torch.float32, torch.float32), (torch.float64, torch.float64),
                                   (torch.float64, torch.float32), (torch.float32, torch.float64)])
@pytest.mark.parametrize("grid,n", [((2, 2, 2), 1), ((17, 5, 33), 255), ((33, 32, 31), 131_072),
                                    ((16, 16, 16), 131_073), ((32, 32, 32), 400_000),
                                    ((32, 32, 32), 400_001), ((100, 101, 102), 300_000)])
def test_direct_gather_equals_interleaved(grid, n, pt, mt):
    import spacecharge as sc
    g = torch.Generator(device=DEV).manual_seed(n)
    x, y, z = (torch.rand(n, generator=g, device=DEV, dtype=torch.float64).mul(2.4).sub(1.2).to(pt)
               for _ in range(3))  # a sixth of each axis lies outside the mesh
    x[0] = 1.0  # the upper face
    if n > 3:
        x[1], y[2], z[3] = float("nan"), float("inf"), -float("inf")
    out = []
    for layout in (0, 1):
        m = sc.Mesh3D(grid, (-1.0,) * 3, (1.0,) * 3, T=mt)
        m.set_field_layout(layout)
        m._ef.copy_(torch.randn(m._ef.numel(), generator=torch.Generator(device=DEV).manual_seed(1),
                                device=DEV, dtype=mt))
        out.append(torch.stack(sc.interpolate_field(m, x, y, z)))
        if n > 1:  # device-resident bounds of the finite particles
            ok = torch.isfinite(x) & torch.isfinite(y) & torch.isfinite(z)
            m.update_bounds(x[ok], y[ok], z[ok])
            out.append(torch.stack(sc.interpolate_field(m, x, y, z)))
    half = len(out) // 2
    for a, b in zip(out[:half], out[half:]):
        assert a.dtype == pt
        assert torch.equal(torch.nan_to_num(a, nan=12345.0), torch.nan_to_num(b, nan=12345.0))
