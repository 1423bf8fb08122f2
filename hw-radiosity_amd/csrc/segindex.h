// Grid over which the explicit matrix's segment visibility is walked
// (device.hip, k_vis_tiles): which triangles can block a segment between two
// of the scene's centroids, listed by cell.
#pragma once

#include <cstdint>
#include <vector>

#include "patch.h"

namespace rgpu {

struct SegIndex {
	bool built = false;
	// cells per axis, a border of empty ones included (cell 1 starts at g0);
	// at most kSegCells in all, so that a bit for each fits a block's LDS
	int r[3] = {0, 0, 0};
	float g0[3] = {0, 0, 0}, h[3] = {1, 1, 1};
	std::vector<int> begin;      // cell (x r[1] + y) r[2] + z -> first item; one more at the end
	std::vector<int> items;      // originals, ascending within a cell
	std::vector<uint32_t> mask;  // bit per cell: has items
};

// The bound on the cells also keeps the walk within what the lists are grown by
// (4e-3 of a cell, below).  The walk adds the parameter of an axis's next wall up
// from the last, so that a wall's place is off by 0.004 of a cell after 512 cells
// and by 0.06 after 2048 (measured).  Along its own axis that only moves the
// moment of a step, and the end of the walk by 3e-5 of the segment, where tests
// stop 1e-4 short of it; a cell skipped for it is one whose part of the segment
// lies within that error of a wall of another axis: in that axis's cells, the
// error times the ratio of the two axes' cells.  An axis of 2048 leaves at most
// 2^18 / (3 * 2048) = 42 for another: 0.06 * 42 / 2048 = 1.2e-3; one of 512, 170:
// 1.3e-3.  With a larger bound the lists would have to grow with it.
constexpr int kSegCells = 1 << 18;

// The index of the originals [0, n) of pool, whose slots are whole (no
// pre-partition); radius: their cull radii (infinite: no bound).  split: the
// segments also run between centroids of triangles cut out of the originals;
// the grid then covers the originals' corners, and none is left out.
//
// Left out otherwise are triangles that no test of any segment between two
// centroids accepts: those whose normal has one component only, in a plane that
// holds the least or the greatest centroid coordinate of its axis (the walls of
// a room).  With X that coordinate, p and q the segment's ends, v = fl(q - p):
// rounding is monotonic, so fl(q - p) is not less than fl(X - p) (not more, for
// the greatest), and the test's quotient fl(fl(X - p) n) / fl(v n) is zero, not
// positive, at least one, or not a number, and so outside (1e-4, 1 - 1e-4).
// Every other triangle is listed in each cell that its bounding box touches,
// grown by 4e-3 of a cell and by 2^-18 of the coordinates (the walk's and the
// tests' rounding), by a whole cell without a cull radius (slivers, whose side
// planes' rounding reaches further).
void build_segment_index(SegIndex &g, const Patch *pool, int n, const float *radius, bool split = false);

}  // namespace rgpu
