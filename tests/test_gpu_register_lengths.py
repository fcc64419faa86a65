"""The register-resident transforms at every length they support.

Each length L serves axes of L/2 nodes and, padded, of every count down to
just above half the next shorter length.  Both ends are solved with the axis
along x, y and z, in every solve mode, and compared with the generic engine
(force_generic_transforms), which the oracle tests pin at the same lengths.

Both engines compute the same transforms in the same type.  Each of the six
passes of a solve is within about 6 eps log2(L) of exact, L <= 512: together
324 eps of the padded spectrum, 7.2e-14 in Float64 and 3.9e-5 in Float32 at
the very worst, a few eps typically (rounding errors add like a random
walk).  The Float32 gate is the suite's 1e-5 and the Float64 one the suite's
1e-12.
"""
import os
import re

import pytest
import torch

from _common import rel_l2

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(REPO, "spacecharge.jl_amd", "csrc", "sc_fft_mix.h")


def _lengths():
    text = open(HEADER).read()
    found = [re.search(r"#define SC_MIX_%s\(X\)([^\n]*)" % k, text).group(1)
             for k in ("SHORT", "LONG", "POW2")]
    return sorted(int(v) for v in re.findall(r"X\((\d+)\)", "".join(found)))


LENGTHS = _lengths()


def test_lengths_are_even_sorted_and_cover_256_nodes():
    assert len(set(LENGTHS)) == len(LENGTHS) and LENGTHS[-1] == 512
    for L in LENGTHS:
        m = L
        for f in (2, 3, 5):
            while m % f == 0:
                m //= f
        assert m == 1 and L % 2 == 0


@pytest.mark.gpu
@pytest.mark.parametrize("T,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
@pytest.mark.parametrize("k", range(len(LENGTHS)), ids=[f"L{v}" for v in LENGTHS])
def test_register_length_matches_generic_engine(k, T, tol):
    import spacecharge as sc
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(LENGTHS[k])
    most = LENGTHS[k] // 2
    least = LENGTHS[k - 1] // 2 + 1 if k else 2
    worst = 0.0
    for n in {most, least}:
        for grid in ((n, 6, 5), (5, n, 6), (6, 5, n)):
            pair = []
            for generic in (False, True):
                m = sc.Mesh3D(grid, (-1e-3, -1e-3, 1e-4), (1e-3, 1.2e-3, 2e-3), T=T, gamma=1.5)
                if generic:
                    m.force_generic_transforms()
                pair.append(m)
            rho = torch.rand(grid, generator=g, device=dev, dtype=T)
            cot = torch.rand(grid + (3,), generator=g, device=dev, dtype=T)
            out = []
            for m in pair:
                m.rho.copy_(rho)
                res = []
                for cath in (False, True):
                    sc.solve(m, at_cathode=cath)
                    res += [m.efield[..., c].cpu().numpy().copy() for c in range(3)]
                    res.append(sc.solve_adjoint(m, cot, at_cathode=cath).cpu().numpy())
                res.append(sc.solve_potential(m).cpu().numpy())
                out.append(res)
            for a, b in zip(*out):
                worst = max(worst, rel_l2(a, b))
    print(f"L={LENGTHS[k]} {T}: register against generic engine {worst:.2e}")
    assert worst <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("grid", [(25, 6, 17), (40, 33, 29), (50, 12, 9)])
def test_float64_particles_keep_a_float32_mesh_on_the_generic_engine(grid):
    """A Float32 mesh that carries Float64 particles is transformed as with
    the generic engine, to the bit (its fields are returned in Float64)."""
    import spacecharge as sc
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(5)
    x, y, z, q = (torch.rand(5000, generator=g, device=dev, dtype=torch.float64) for _ in range(4))
    out = []
    for generic in (False, True):
        m = sc.Mesh3D(grid, x, y, z, T=torch.float32)
        if generic:
            m.force_generic_transforms()
        sc.deposit(m, x, y, z, q)
        sc.solve(m)
        out.append(torch.stack(sc.interpolate_field(m, x, y, z)))
    assert out[0].dtype == torch.float64 and torch.equal(out[0], out[1])


# Green builds of the fused kernel: several z planes per workgroup and a ragged
# last group, rows that end inside a workgroup's strip, and (last) an F lattice
# beyond the 256 MB last-level cache.
@pytest.mark.gpu
@pytest.mark.parametrize("T,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
@pytest.mark.parametrize("grid", [(3, 2, 2), (9, 30, 250), (12, 7, 199), (100, 9, 31), (16, 16, 300),
                                  (64, 512, 350)])
def test_fused_green_build_matches_separate_passes(grid, T, tol):
    import spacecharge as sc
    dev = torch.device("cuda:0")
    rho = torch.rand(grid, generator=torch.Generator(device=dev).manual_seed(9), device=dev, dtype=T)
    worst = 0.0
    for cath in (False, True):
        out = []
        for generic in (False, True):
            m = sc.Mesh3D(grid, (-1e-3, -1e-3, 1e-4), (1e-3, 1.2e-3, 2e-3), T=T, gamma=2.0)
            if generic:
                m.force_generic_transforms()
            m.rho.copy_(rho)
            sc.solve(m, at_cathode=cath)
            out.append(m.efield.cpu().numpy())
            del m
        worst = max(worst, max(rel_l2(out[0][..., c], out[1][..., c]) for c in range(3)))
    print(f"fused Green build {grid} {T}: {worst:.2e}")
    assert worst <= tol
