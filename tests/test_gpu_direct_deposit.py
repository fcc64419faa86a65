"""The deposit without binning (meshes of few tiles) at the edges of its range.

Against the oracle and the binned chain (any tiling other than the default
selects it).  A node's sum of k contributions, each rounded once in the
particle arithmetic, then summed in Float64: Float64 meshes agree to a few
times 1e-16 sqrt(k), gated at the suite's 1e-13; Float32 meshes round the
Float64 sum once (6e-8) after contributions formed in Float32 arithmetic as
the oracle forms them: gated at the suite's 1e-5 against the Float64 oracle and
to the bit against the binned chain (the same fixed-point contributions).
"""
import numpy as np
import pytest
import torch

import oracle as orc
from _common import mesh_to_np, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# (grid, particles): one tile to 64, a slice and one more, a workgroup's lanes
# and one more, odd counts, one particle
CASES = [((2, 2, 2), 1), ((16, 16, 16), 511), ((17, 17, 17), 513), ((18, 17, 16), 8192),
         ((17, 9, 17), 300_001), ((33, 33, 33), 8193), ((33, 18, 49), 64_001),
         ((48, 48, 48), 155_000), ((64, 64, 64), 65_536), ((65, 65, 65), 20_011)]


def _bunch(n, seed, dtype, spread):
    rng = np.random.default_rng(seed)
    p = rng.standard_normal((3, n)) * spread
    q = rng.uniform(-0.5, 1.0, n) * 1e-9
    return [torch.as_tensor(a, dtype=dtype, device=DEV) for a in (*p, q)]


@pytest.mark.parametrize("pt,mt", [(torch.float32, torch.float32), (torch.float64, torch.float64),
                                   (torch.float64, torch.float32), (torch.float32, torch.float64)])
@pytest.mark.parametrize("grid,n", CASES)
def test_direct_deposit_matches_oracle_and_binned(grid, n, pt, mt):
    import spacecharge as sc
    # a third of the particles lie outside the mesh (clamped, extrapolating)
    # in the odd cases, none in the even ones
    spread = 1.0 if n % 2 else 0.2
    x, y, z, q = _bunch(n, n + grid[0], pt, spread)
    meshes = [sc.Mesh3D(grid, (-1.0,) * 3, (1.0,) * 3, T=mt) for _ in range(2)]
    meshes[1].set_deposit_tiling(12, 11)
    for m in meshes:
        sc.deposit(m, x, y, z, q)
        once = m.rho.clone()
        sc.deposit(m, x, y, z, q, clear=False)
        assert rel_l2(m.rho.cpu().numpy(), 2 * once.cpu().numpy()) <= (1e-6 if mt == torch.float32 else 1e-14)
        m.rho.copy_(once)
    host = [a.double().cpu().numpy() for a in (x, y, z, q)]
    m = meshes[0]
    ref = orc.deposit(*host, grid, m.min_bounds, m.delta)
    got, binned = (mesh_to_np(k._rho, grid) for k in meshes)
    scale = np.linalg.norm(ref.ravel())
    e = np.linalg.norm((got.astype(np.float64) - ref).ravel()) / scale
    b = np.linalg.norm((got.astype(np.float64) - binned).ravel()) / scale
    print(f"direct deposit {grid} n={n} {pt} {mt}: oracle {e:.2e} binned {b:.2e}")
    single = pt == torch.float32 or mt == torch.float32
    assert e <= (1e-5 if single else 1e-13)
    assert np.array_equal(got, binned) if mt == torch.float32 else b <= 1e-13


@pytest.mark.parametrize("grid", [(16, 16, 16), (33, 20, 17)])
def test_direct_deposit_nonfinite_and_denormal_charges(grid):
    """Infinite, NaN and tiny charges take the Float64 accumulator."""
    import spacecharge as sc
    x, y, z, q = _bunch(4000, 3, torch.float32, 0.2)
    for bad in (float("inf"), float("nan"), 0.0):
        p = q.clone()
        if bad == 0.0:
            p.fill_(1e-44)
        else:
            p[1234] = bad
        out = []
        for tiling in (None, (12, 11)):
            m = sc.Mesh3D(grid, (-1.0,) * 3, (1.0,) * 3, T=torch.float32)
            if tiling:
                m.set_deposit_tiling(*tiling)
            sc.deposit(m, x, y, z, p)
            out.append(m.rho.cpu().numpy())
        assert np.array_equal(np.isfinite(out[0]), np.isfinite(out[1]))
        ok = np.isfinite(out[0])
        assert np.allclose(out[0][ok], out[1][ok], rtol=1e-6, atol=1e-44 if bad == 0.0 else 1e-16)


@pytest.mark.parametrize("T", [torch.float32, torch.float64])
@pytest.mark.parametrize("grid", [(16, 16, 16), (33, 20, 17)])
def test_direct_deposit_three_channels_and_device_bounds(grid, T):
    """The cotangent deposit (three channels) and device-resident bounds."""
    import spacecharge as sc
    x, y, z, q = _bunch(7001, 4, T, 0.2)
    g = [torch.randn_like(x) for _ in range(3)]
    out = []
    for tiling in (None, (12, 11)):
        m = sc.Mesh3D(grid, (-1.0,) * 3, (1.0,) * 3, T=T)
        if tiling:
            m.set_deposit_tiling(*tiling)
        m.update_bounds(x, y, z)
        sc.deposit(m, x, y, z, q)
        rho = m.rho.cpu().numpy().copy()
        gef = sc.interpolate_adjoint(m, x, y, z, *g)[0]
        out.append((rho, gef.cpu().numpy()))
    for a, b in zip(*out):
        assert np.array_equal(a, b) if T == torch.float32 else rel_l2(a, b) <= 1e-13
