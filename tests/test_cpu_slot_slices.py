"""The slot arrays hold a slice for every wavefront of every tile.

The BVD pass reads the slot faces of a wavefront's slice before it knows which
of its cells exist, so the last tile of 128 or 256 cells needs the slices of
wavefronts that lie wholly past the last cell, and finds no slot (0) there.
The layout code runs on the CPU, over cell counts on both sides of each
wavefront of a last tile; the index is the kernel's."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "afar_cudaeuler2dmixo3rk3solver_amd", "csrc")

PROGRAM = r"""
#include <cstdio>
#include "layout.h"
using namespace afar;
int main() {
    int bad = 0, checked = 0;
    for (int nx : {3, 9, 16, 20, 22, 25, 32}) {
        const double inflow[4] = {1 / 1.4, 2.0, 0.0, 1.0};
        Mesh m = build_mesh(generate_corner(nx, 7, 1.0, 0.5, 0.15, 1, 0.5, 15.0, inflow, 2), true);
        Schemes sc;
        Precomputed pc = precompute(m, sc);
        std::vector<double> W0(4 * (size_t)m.nc, 1.0);
        RefArrays ra = make_ref_arrays(m, pc, W0.data(), sc.R, sc.Cv);
        for (int tile : {64, 128, 256}) {
            const DevLayout L = make_dev_layout(ra, tile);
            const int last = (L.ntiles - 1) * tile;  // the last tile's first cell
            for (int t = 0; t < tile; ++t)
                for (int k = 0; k < L.maxC; ++k) {
                    const size_t slice = (unsigned)(last + 64 * (t >> 6)) >> 6;
                    const size_t i = slice * L.maxC * 64 + k * 64 + (t & 63);
                    ++checked;
                    if (i >= L.slot_face.size()) ++bad;
                    else if (last + t >= L.nc && L.slot_face[i] != 0) ++bad;
                }
        }
    }
    printf("%d of %d\n", bad, checked);
    return bad != 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_wavefront_has_its_slice(tmp_path):
    src, exe = tmp_path / "slices.cpp", str(tmp_path / "slices")
    src.write_text(PROGRAM)
    cmd = ["g++", "-O1", "-std=c++17", "-I", CSRC, "-o", exe, str(src)] + [
        os.path.join(CSRC, f) for f in ("mesh.cpp", "precompute.cpp", "layout.cpp")] + ["-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
