"""The grid of the segment visibility (segindex.h) on the host: a bit per cell
has to fit a block's LDS, and a triangle no larger than a cell is in few cells'
lists, whatever the scene's size, detail and distance from the origin."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "hw-radiosity_amd", "csrc")

# a frame of eight triangles around 400 small ones, off from the origin along x
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "segindex.h"
using namespace rgpu;
int main(int, char **argv)
{
	const double off = std::atof(argv[1]), small = std::atof(argv[2]);
	std::vector<Patch> pool;
	std::vector<float> radius;
	auto add = [&](double x, double y, double z, double s) {
		const double q[3][3] = {{x + off, y, z}, {x + off, y + s, z}, {x + off, y, z + s}};
		Patch t{};
		for (int v = 0; v < 3; v++)
			for (int k = 0; k < 3; k++) t.p[v][k] = (float)q[v][k];
		centroid(t.p, t.c);
		t.n[0] = t.n[1] = (float)(s * s);
		t.area = (float)(s * s / 2);
		pool.push_back(t);
		radius.push_back((float)s);
	};
	for (int i = 0; i < 8; i++) add(i & 1 ? 10 : 0, i & 2 ? 9 : 0, i & 4 ? 9 : 0, 1);
	for (int i = 0; i < 400; i++) add(5, 4 + small * (i % 20), 4 + small * (i / 20), small);
	SegIndex g;
	build_segment_index(g, pool.data(), (int)pool.size(), radius.data());
	std::printf("%lld %d %zu %zu %d %g\n", (long long)g.r[0] * g.r[1] * g.r[2], kSegCells, g.begin.size(), g.mask.size(),
	            g.begin.back(), g.h[1] < g.h[2] ? g.h[1] : g.h[2]);
	return 0;
}
"""


@pytest.fixture(scope="module")
def grid(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    d = tmp_path_factory.mktemp("segindex")
    (d / "main.cpp").write_text(MAIN)
    r = subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, str(d / "main.cpp"), os.path.join(CSRC, "segindex.cpp"),
                        "-o", str(d / "grid")], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
    return str(d / "grid")


@pytest.mark.parametrize("small", ["0.3", "0.01", "1e-6"])
@pytest.mark.parametrize("off", ["0", "1e5", "3e6", "1e7", "1e9"])
def test_cells_stay_within_their_bound(grid, off, small):
    r = subprocess.run([grid, off, small], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0
    cells, most, begins, words, items = (int(x) for x in r.stdout.split()[:5])
    h = float(r.stdout.split()[5])  # cells along y and z
    assert 27 <= cells <= most
    assert begins == cells + 1 and words == (cells + 31) // 32
    # the lists are grown by at most a cell each way: a triangle of size s
    # lies in s / h + 3 cells along y and z, and in 4 along x
    assert items <= 4 * (400 * (float(small) / h + 3) ** 2 + 8 * (1 / h + 3) ** 2)
