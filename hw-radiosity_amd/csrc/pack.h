// Host side of the upload: the order in which the device takes receivers.
#pragma once

#include <cstddef>

#include "patch.h"

namespace rgpu {

// order[0..n) = the slots sorted by the Z-order (Morton) code of their
// centroids on a 2^10 grid over [G0, G1], ties by slot; a permutation.
void spatial_order(const Patch *pool, int n, const float *G0, const float *G1, int *order);

// memcpy, by several threads from 256 KB up (one thread copies at about 30
// GB/s, the link to the device takes 55, and the pages of a fresh array are
// first touched here)
void copy_bytes(void *dst, const void *src, size_t bytes);

}  // namespace rgpu
