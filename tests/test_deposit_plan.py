"""The deposit's scratch, on the host: what one deposit reserves holds every later
deposit of at most as many particles and channels on the same mesh, by the direct
path and by the binned chain (batched calls, a tiling of the mesh's own, the sort
permutation).  A deposit that needed more would move the buffers whose addresses a
captured graph holds, or allocate inside a capture.

The arithmetic is sc_deposit_plan.h itself, compiled for the host."""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "spacecharge.jl_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "sc_deposit_plan.h"
using namespace sc;
int main()
{
    const int tiles[] = {1, 2, 3, 5, 8, 12, 18, 27, 36, 48, 54, 63, 64, 65, 125, 512};
    long bad = 0, checked = 0, direct = 0;
    for (int T : tiles)
        for (int f32 = 0; f32 < 2; ++f32)
            for (int nchan = 1; nchan <= 3; nchan += 2)
                for (double nf = 1; nf < 2.0e7; nf = nf * 1.17 + 1) {
                    const int64_t n = (int64_t)nf;
                    const DepositNeed have = deposit_need(n, T, f32, nchan, 13, 12);
                    for (double sf = 1; (int64_t)sf <= n; sf = sf * 1.11 + 1) {
                        const int64_t k = (int64_t)sf;
                        for (int c = 1; c <= nchan; c += 2) {
                            const DepositNeed b = binned_need(k, T, 13, 12);
                            bool ok = b.chunks <= have.chunks && b.cmat <= have.cmat;
                            if (k <= direct_most(T, f32, c)) {
                                const DepositNeed d = direct_need(k, T, c);
                                ok = ok && d.chunks <= have.chunks && d.cmat <= have.cmat;
                                // slices of at most 2^13 particles: 16-bit list entries
                                const int G = direct_slices(k, T);
                                ok = ok && G >= 1 && (k + G - 1) / G <= (1 << kDirectLog2);
                                ++direct;
                            }
                            ++checked;
                            if (!ok && bad++ < 10)
                                std::printf("T=%d f32=%d: %ld in %d channels after %ld in %d\n", T, f32,
                                            (long)k, c, (long)n, nchan);
                        }
                    }
                }
    std::printf("%ld deposits checked, %ld of them direct, %ld too large\n", checked, direct, bad);
    return bad || !direct;
}
"""


def test_scratch_of_a_deposit_holds_every_smaller_one(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-O1", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
