#include "segindex.h"

#include <algorithm>
#include <cmath>

namespace rgpu {

void build_segment_index(SegIndex &g, const Patch *pool, int n, const float *radius, bool split)
{
	float lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
	for (int i = 0; i < n; i++)
		for (int k = 0; k < 3; k++) {
			const float (&p)[3][3] = pool[i].p;
			const float c = pool[i].c[k];
			const float mn = split ? std::min({p[0][k], p[1][k], p[2][k]}) : c, mx = split ? std::max({p[0][k], p[1][k], p[2][k]}) : c;
			lo[k] = i ? std::min(lo[k], mn) : mn;
			hi[k] = i ? std::max(hi[k], mx) : mx;
		}
	std::vector<int> cand;
	double area = 0.0;
	for (int i = 0; i < n; i++) {
		const Patch &t = pool[i];
		bool never = false;
		for (int k = 0; k < 3 && !split; k++)
			never |= t.n[(k + 1) % 3] == 0.0f && t.n[(k + 2) % 3] == 0.0f && (t.c[k] == lo[k] || t.c[k] == hi[k]);
		if (never) continue;
		cand.push_back(i);
		area += t.area;
	}
	// cells of 1.5 times the side of a mean candidate (as half a square), as far
	// as the number of cells allows (rooms of 3000, 9000 and 20000 patches, ms of
	// walk and matrix: 0.66, 3.7, 16.8 at 0.7; 0.54, 3.1, 14.0 at 1; 0.61, 2.9,
	// 12.6 at 1.5; 0.58, 3.3, 12.8 at 2; 0.69, 3.8, 14.9 at 3)
	double ext = 0.0, mag = 0.0;
	for (int k = 0; k < 3; k++) {
		ext = std::max(ext, (double)hi[k] - lo[k]);
		mag = std::max({mag, std::fabs((double)lo[k]), std::fabs((double)hi[k])});
	}
	double side = cand.empty() ? ext : 1.5 * std::sqrt(2.0 * area / cand.size());
	if (!(side > 0.0) || !std::isfinite(side)) side = ext > 0.0 ? ext : 1.0;
	// ... nor less than twice what the lists are grown by (below), so that scenes
	// far from the origin, whose coordinates round by much of a cell, do not list
	// each triangle in all the cells around it
	const double grow = 0x1p-18 * (mag + ext);
	side = std::max(side, 2.0 * grow);
	// the grid's extent along an axis: that of the centroids and their rounding
	auto extent = [&](int k) { return ((double)hi[k] - lo[k]) * (1.0 + 2e-3) + mag * 0x1p-20 + 1e-30; };
	auto cells = [&](double s) {
		double p = 1.0;
		for (int k = 0; k < 3; k++) p *= std::ceil(extent(k) / s) + 3.0;
		return p;
	};
	while (cells(side) > kSegCells) side *= 1.05;
	for (int k = 0; k < 3; k++) {
		const double e = extent(k);
		const int inner = std::max(1, (int)std::ceil(e / side));
		g.r[k] = inner + 2;
		g.h[k] = (float)(e / inner);
		g.g0[k] = (float)(((double)lo[k] + hi[k]) * 0.5 - e * 0.5);
	}
	const size_t nc = (size_t)g.r[0] * g.r[1] * g.r[2];
	// the cells [a, b] of every axis that candidate i touches; false: none
	auto range = [&](int i, int (&a)[3], int (&b)[3]) {
		const Patch &t = pool[i];
		const bool wide = !std::isfinite(radius[i]);
		for (int k = 0; k < 3; k++) {
			const double mn = std::min({t.p[0][k], t.p[1][k], t.p[2][k]}), mx = std::max({t.p[0][k], t.p[1][k], t.p[2][k]});
			const double slack = wide ? 1.0 : 4e-3;
			const double fa = std::floor((mn - grow - g.g0[k]) / g.h[k] - slack), fb = std::floor((mx + grow - g.g0[k]) / g.h[k] + slack);
			if (fb < 0.0 || fa > g.r[k] - 3) return false;
			a[k] = 1 + (int)std::max(0.0, fa);
			b[k] = 1 + (int)std::min((double)(g.r[k] - 3), fb);
		}
		return true;
	};
	g.begin.assign(nc + 1, 0);
	for (int pass = 0; pass < 2; pass++) {
		for (int i : cand) {
			int a[3], b[3];
			if (!range(i, a, b)) continue;
			for (int x = a[0]; x <= b[0]; x++)
				for (int y = a[1]; y <= b[1]; y++)
					for (int z = a[2]; z <= b[2]; z++) {
						int &c = g.begin[((size_t)x * g.r[1] + y) * g.r[2] + z];
						if (pass) g.items[c] = i;
						c++;
					}
		}
		if (pass == 0) {  // counts -> first items
			int run = 0;
			for (size_t c = 0; c <= nc; c++) {
				const int k = g.begin[c];
				g.begin[c] = run;
				run += k;
			}
			g.items.resize(run);
		}
	}
	// the fill left each cell's end in begin: shift back to its start
	for (size_t c = nc; c > 0; c--) g.begin[c] = g.begin[c - 1];
	g.begin[0] = 0;
	g.mask.assign((nc + 31) / 32, 0);
	for (size_t c = 0; c < nc; c++)
		if (g.begin[c + 1] > g.begin[c]) g.mask[c >> 5] |= 1u << (c & 31);
	g.built = true;
}

}  // namespace rgpu
