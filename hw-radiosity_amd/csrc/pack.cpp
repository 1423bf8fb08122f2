#include "pack.h"

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

void copy_bytes(void *dst, const void *src, size_t bytes)
{
	constexpr size_t kSlice = (size_t)128 << 10;
	if (bytes < 2 * kSlice) {
		std::memcpy(dst, src, bytes);
		return;
	}
	const long slices = (long)((bytes + kSlice - 1) / kSlice);
	// always the same number of threads: a team that changes its size ends and
	// starts threads, 30 us and more a call.  With a thread per slice instead, us:
	// 1.5 MB to the device 104 (68 so), 4 MB back 222 (154); 65536 rays cast 260
	// (180), where copies by the runtime itself take 240.  Eight, not the 16 of
	// the engine's other loops, though the scene read after a copy then has to
	// start threads (1445 us, 1335 after 16): beside torch's own team, 16 threads
	// took 1980 us for a cast of 10^6 rays (1840), 4560 for 192 columns on 7777
	// patches (4200).  Eight of the engine's own, asleep between calls, read that
	// scene in 1400 but cast 100000 rays after it in 400 to 740 (285)
#pragma omp parallel for schedule(static) num_threads(8)
	for (long k = 0; k < slices; k++) {
		const size_t o = (size_t)k * kSlice;
		std::memcpy((char *)dst + o, (const char *)src + o, bytes - o < kSlice ? bytes - o : kSlice);
	}
}

}  // namespace rgpu
