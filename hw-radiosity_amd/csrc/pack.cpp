#include "pack.h"

#include <omp.h>
#include <parallel/algorithm>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

namespace rgpu {

namespace {
// the bits of x spread to every third position
inline uint32_t spread3(uint32_t x)
{
	x &= 0x3ffu;
	x = (x | (x << 16)) & 0x030000ffu;
	x = (x | (x << 8)) & 0x0300f00fu;
	x = (x | (x << 4)) & 0x030c30c3u;
	x = (x | (x << 2)) & 0x09249249u;
	return x;
}
}  // namespace

void spatial_order(const Patch *pool, int n, const float *G0, const float *G1, int *order)
{
	std::vector<uint64_t> key(n);
#pragma omp parallel for schedule(static)
	for (int i = 0; i < n; i++) {
		uint32_t code = 0;
		for (int k = 0; k < 3; k++) {
			const double span = (double)G1[k] - (double)G0[k];
			double u = span > 0 ? ((double)pool[i].c[k] - (double)G0[k]) / span * 1024.0 : 0.0;
			if (!(u >= 0.0)) u = 0.0;  // NaN too
			if (u > 1023.0) u = 1023.0;
			code |= spread3((uint32_t)u) << k;
		}
		key[i] = ((uint64_t)code << 32) | (uint32_t)i;
	}
	__gnu_parallel::sort(key.begin(), key.end());
#pragma omp parallel for schedule(static)
	for (int i = 0; i < n; i++) order[i] = (int)(uint32_t)key[i];
}

// The team that the engine's other loops use, so that none changes its size: that
// ends and starts threads.  us, 16 threads on 16 CPUs, a team of one thread per
// slice (at most eight), of eight, of all: 1.5 MB to the device 104, 68, 69, 4 MB
// back 222, 154, 155; 65536 rays cast 260, 180, 179 (240 by the runtime's own
// copies); the scene read between two casts, which has to start the threads
// again, 1445 after eight, 1335 after all, as without any copy.  Where that team
// is wide, or larger than the CPUs, eight: 64 threads on 16 CPUs took 284 us for
// the first 1.1 MB (62).
static int copy_team()
{
	const int all = omp_get_max_threads(), cpus = omp_get_num_procs();
	return all <= 32 && all <= cpus ? all : cpus < 8 ? cpus : 8;
}

void copy_bytes(void *dst, const void *src, size_t bytes)
{
	constexpr size_t kSlice = (size_t)128 << 10;
	if (bytes < 2 * kSlice) {
		std::memcpy(dst, src, bytes);
		return;
	}
	const long slices = (long)((bytes + kSlice - 1) / kSlice);
#pragma omp parallel for schedule(static) num_threads(copy_team())
	for (long k = 0; k < slices; k++) {
		const size_t o = (size_t)k * kSlice;
		std::memcpy((char *)dst + o, (const char *)src + o, bytes - o < kSlice ? bytes - o : kSlice);
	}
}

}  // namespace rgpu
