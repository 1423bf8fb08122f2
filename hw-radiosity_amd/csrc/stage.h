// Pinned staging for the copies between a caller's pageable arrays and the
// device, one per handle (the handle's own thread and stream use it).
//
// The runtime's copy of pageable memory costs 0.4 us per KB between about 16
// KB and 1 MB (measured, us, host to device: 24 KB 16, 96 KB 44, 512 KB 210;
// from pinned memory 9, 10, 18, and the memcpy into it 0.3, 1, 9), and at
// larger sizes it stays well below the link (12 MB: 359 us to the device, 739
// back, against 229 from and to pinned memory).  Small copies go through 1 MB
// of pinned memory made with the handle (0.05 ms), larger ones in chunks
// through four more made on their first use (0.3 ms), the host's side of a
// chunk copied by several threads (copy_bytes) while others are on their way.
// Include inside the translation unit's anonymous namespace (after HIP_OK).
#pragma once

struct Stage {
	static constexpr size_t kSmall = (size_t)1 << 20;  // pinned bytes for small copies
	// Arrays up to this many bytes, in the pinned memory for small copies, are
	// read and written over the link by the kernels that use them, where a copy's
	// launch and the wait for it cost more than the slower access.  us, copied and
	// direct: a gather of n = 1000, 2000, 4000, 8000 with 3 columns 202, 212, 284,
	// 756 and 160, 180, 262, 733, of n = 2000 with 24 (750 KB in) 275 and 270; 10,
	// 3000, 16000 rays cast 44, 50, 71 and 32, 36, 51.
	static constexpr size_t kDirect = (size_t)768 << 10;
	static constexpr size_t kChunk = (size_t)1 << 20;  // of a large copy
	static constexpr int kDepth = 4;                   // chunks on their way
	unsigned char *p = nullptr, *q = nullptr;
	size_t off = 0, keep = 0;  // bytes of p in use; those of room(), which copies leave alone
	hipEvent_t ev[kDepth] = {};
	// per-block statistics that kernels write to host memory directly (read
	// after the stream is synchronised: no copy to wait for)
	double *stats = nullptr;
	size_t nstats = 0;

	Stage() = default;
	Stage(const Stage &) = delete;
	Stage &operator=(const Stage &) = delete;
	~Stage()
	{
		for (hipEvent_t e : ev)
			if (e) (void)hipEventDestroy(e);
		if (p) (void)hipHostFree(p);
		if (q) (void)hipHostFree(q);
		if (stats) (void)hipHostFree(stats);
	}
	int init(std::string &err)
	{
		if (p) return 0;
		for (hipEvent_t &e : ev) HIP_OK(hipEventCreateWithFlags(&e, hipEventDisableTiming), "event");
		HIP_OK(hipHostMalloc((void **)&p, kSmall, hipHostMallocDefault), "pinned staging");
		return 0;
	}
	int large(std::string &err)
	{
		if (!q) HIP_OK(hipHostMalloc((void **)&q, kDepth * kChunk, hipHostMallocDefault), "pinned staging");
		return 0;
	}
	// room for n doubles of statistics; no kernel may be writing to them
	int stat_room(size_t n, std::string &err)
	{
		if (n <= nstats) return 0;
		if (stats) (void)hipHostFree(stats);
		stats = nullptr;
		nstats = 0;
		HIP_OK(hipHostMalloc((void **)&stats, n * sizeof(double), hipHostMallocDefault), "pinned statistics");
		nstats = n;
		return 0;
	}
	// the next calls' copies start at the buffer's beginning: none of the
	// earlier ones may be in flight (the stream was synchronised), and what
	// room() gave out is done with
	void begin() { off = keep = 0; }
	// queues a copy to the device; src may be reused at once.  grow = false
	// (callers that must not allocate): a large copy goes directly where the
	// chunks are not there yet, and src is free once the stream is synchronised
	int up(void *dst, const void *src, size_t bytes, hipStream_t st, std::string &err, bool grow = true)
	{
		if (bytes == 0) return 0;
		if (bytes <= kSmall - keep) {
			if (off + bytes > kSmall) {
				HIP_OK(hipStreamSynchronize(st), "upload");
				off = keep;
			}
			std::memcpy(p + off, src, bytes);
			HIP_OK(hipMemcpyAsync(dst, p + off, bytes, hipMemcpyHostToDevice, st), "upload");
			off += (bytes + 255) / 256 * 256;
			return 0;
		}
		if (!q && !grow) {
			HIP_OK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st), "upload");
			return 0;
		}
		if (large(err)) return -1;
		HIP_OK(hipStreamSynchronize(st), "upload");  // the chunks' earlier copies
		for (size_t c = 0; c * kChunk < bytes; c++) {
			const size_t o = c * kChunk, b = std::min(kChunk, bytes - o);
			unsigned char *h = q + (c % kDepth) * kChunk;
			if (c >= (size_t)kDepth) HIP_OK(hipEventSynchronize(ev[c % kDepth]), "upload");
			copy_bytes(h, (const unsigned char *)src + o, b);
			HIP_OK(hipMemcpyAsync((unsigned char *)dst + o, h, b, hipMemcpyHostToDevice, st), "upload");
			HIP_OK(hipEventRecord(ev[c % kDepth], st), "upload");
		}
		return 0;
	}
	// room for bytes that kernels read or write in the pinned memory themselves
	// (until begin()), or null where a copy is the better way
	unsigned char *room(size_t bytes)
	{
		if (bytes > kDirect || off + bytes > kSmall) return nullptr;
		unsigned char *h = p + off;
		keep = off = std::min(kSmall, off + (bytes + 255) / 256 * 256);
		return h;
	}
	// copies src's bytes from the device into consecutive parts of the host's;
	// they are complete on return (the stream is synchronised up to the copy)
	struct Part {
		void *dst;
		size_t bytes;
	};
	int down_parts(const void *src, const Part *part, int parts, hipStream_t st, std::string &err, bool grow = true)
	{
		size_t bytes = 0;
		for (int k = 0; k < parts; k++) bytes += part[k].bytes;
		if (bytes == 0) return 0;
		int k = 0;
		size_t done = 0;  // bytes of part k already copied
		auto scatter = [&](const unsigned char *h, size_t n) {
			while (n > 0) {
				while (done == part[k].bytes) {
					k++;
					done = 0;
				}
				const size_t b = std::min(n, part[k].bytes - done);
				copy_bytes((unsigned char *)part[k].dst + done, h, b);
				h += b;
				n -= b;
				done += b;
			}
		};
		if (bytes <= kSmall - keep) {
			if (off + bytes > kSmall) {
				HIP_OK(hipStreamSynchronize(st), "download");
				off = keep;
			}
			HIP_OK(hipMemcpyAsync(p + off, src, bytes, hipMemcpyDeviceToHost, st), "download");
			HIP_OK(hipStreamSynchronize(st), "download");
			scatter(p + off, bytes);
			return 0;
		}
		if (!q && !grow) {
			const unsigned char *s = static_cast<const unsigned char *>(src);
			for (k = 0; k < parts; s += part[k].bytes, k++)
				HIP_OK(hipMemcpyAsync(part[k].dst, s, part[k].bytes, hipMemcpyDeviceToHost, st), "download");
			HIP_OK(hipStreamSynchronize(st), "download");
			return 0;
		}
		if (large(err)) return -1;
		HIP_OK(hipStreamSynchronize(st), "download");  // the chunks' earlier copies
		const size_t nc = (bytes + kChunk - 1) / kChunk;
		auto issue = [&](size_t c) -> int {
			HIP_OK(hipMemcpyAsync(q + (c % kDepth) * kChunk, (const unsigned char *)src + c * kChunk,
			                      std::min(kChunk, bytes - c * kChunk), hipMemcpyDeviceToHost, st), "download");
			HIP_OK(hipEventRecord(ev[c % kDepth], st), "download");
			return 0;
		};
		for (size_t c = 0; c < std::min<size_t>(nc, kDepth); c++)
			if (issue(c)) return -1;
		for (size_t c = 0; c < nc; c++) {
			HIP_OK(hipEventSynchronize(ev[c % kDepth]), "download");
			scatter(q + (c % kDepth) * kChunk, std::min(kChunk, bytes - c * kChunk));
			if (c + kDepth < nc && issue(c + kDepth)) return -1;
		}
		return 0;
	}
	int down(void *dst, const void *src, size_t bytes, hipStream_t st, std::string &err, bool grow = true)
	{
		const Part one{dst, bytes};
		return down_parts(src, &one, 1, st, err, grow);
	}
};
