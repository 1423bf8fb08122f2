// Linear radiosity solvers on an explicit form-factor matrix (see linear.h).
//
// HBM layout
//   F32   ld x ld floats, row-major, zero padded (ld = n rounded up to 256);
//         the matrix of record: FP64 residuals and the FP32 solvers read it.
//   F16 / BF16  s * F in MFMA fragment order, made on demand: the matrix is
//         cut into 16 x 32 tiles, tile (rb, kb) at ((rb * ld/32) + kb) * 512
//         elements, and inside a tile lane l's 8 elements (row rb*16 + l%16,
//         columns kb*32 + 8*(l/16) .. +7) at l*8.  One wave-wide 16-byte load
//         per lane fetches a whole A fragment as 1 KB of contiguous HBM.
//         s is a power of two that lifts the largest |F| to ~2^14 for FP16
//         (form factors of 1e-6 would otherwise be FP16 subnormals) and 1 for
//         BF16; the product is scaled back by 1/s exactly.
//   XT    the low-precision iterate, nrhs (rounded up to 16) x ld, in the
//         same fragment order (it is the MFMA B operand).
//
// MFMA (v_mfma_f32_16x16x32_{f16,bf16}, gfx950): lane l supplies
// A[l%16][8*(l/16)+j] and B[8*(l/16)+j][l%16], j = 0..7, and receives
// D[4*(l/16)+j][l%16], j = 0..3.  A wave owns 16*RT rows and all 16*CT
// right-hand-side columns, so F is read from HBM once per sweep; split-K S
// spreads the K loop over S waves of a block (k_sweep) or, with 8 or 12 column
// tiles and RT 2 or 4, over S blocks (k_gemm_dma), whose partial tiles are
// summed in a fixed order (results do not depend on timing).  (RT, S) go by the
// size (sweep_tile), unless the caller had the tuner time every tile or set one.
#include "linear.h"

#include "pack.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <map>
#include <type_traits>
#include <vector>

namespace rgpu {
namespace {

#include "lin_common.h"
#include "stage.h"

// One sweep in one launch
template <typename E, int RT, int CT>
__global__ __launch_bounds__(kSweepWaves * 64) void k_sweep(const E *__restrict__ A, const E *__restrict__ XT, int ld,
                                                            int S, bool cached, SweepOut<E> o)
{
	__shared__ f4 red[kSweepWaves * RT * CT * 64];
	sweep_rows<E, RT, CT>(A, XT, ld, S, cached, blockIdx.x, red, o);
}

// Wide right-hand sides (NCT = 8 or 12 column tiles) with the operands
// staged by LDS DMA.  A block is eight waves over 256 rows: WC = 1 gives each
// wave 16 RT = 32 rows and every column, WC = 2 gives it 64 rows and half the
// columns, which cuts the block's LDS reads per k-block from 112 to 80 KB (a
// wave with 64 rows and every column would need its accumulators in AGPRs,
// which the register allocator then copies every k-block).  Each k-block's A
// fragments (1 KB each, those of a row group split over its WC waves) and B
// fragments (spread over the waves) go straight from HBM into a ring of NS
// LDS slots (global_load_lds_dwordx4: no registers held while in flight),
// NS - 1 k-blocks ahead of the MFMAs: 64 KB of A per CU in flight, where a
// register pipeline holds 32 KB.  The compiler treats any LDS read as
// dependent on every LDS DMA in flight and would drain them all before it,
// so the slot is read by inline assembly (its own lgkmcnt wait inside;
// early-clobber outputs, so no read overwrites the address of a later one)
// after an explicit vmcnt wait for this k-block's DMAs and a barrier; every
// trip issues the same DMAs per wave (the index is clamped past the chunk's
// end; those slots are never read), so the vmcnt bound holds to the last
// trip.  The second wave on each SIMD (waves 4-7) runs half a k-block
// behind: after each barrier it multiplies the previous k-block while the
// first wave reads, then reads while the first wave multiplies (0.433 ->
// 0.389 ms for 192 columns at n = 32768, where all eight waves had read and
// then multiplied in step).
// cache policy operand of global_load_lds: nt (non-temporal)
constexpr int kCpolNT = 2;

template <int N>
__device__ __forceinline__ void wait_vmcnt()
{
	static_assert(N >= 0 && N < 64, "vmcnt is six bits");
	asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// RT A fragments (offsets 0, 1024, ...) from ab, then CT B fragments from bb,
// completed before the block ends
#define RGPU_DS1(i, base, off) "ds_read_b128 %" #i ", %" #base " offset:" #off "\n"
template <int RT, int CT, typename V>
__device__ __forceinline__ void read_slot(V (&a)[RT], V (&b)[CT], unsigned ab, unsigned bb)
{
	if constexpr (RT == 2 && CT == 12) {
		asm volatile(RGPU_DS1(0, 14, 0) RGPU_DS1(1, 14, 1024) RGPU_DS1(2, 15, 0) RGPU_DS1(3, 15, 1024)
		             RGPU_DS1(4, 15, 2048) RGPU_DS1(5, 15, 3072) RGPU_DS1(6, 15, 4096) RGPU_DS1(7, 15, 5120)
		             RGPU_DS1(8, 15, 6144) RGPU_DS1(9, 15, 7168) RGPU_DS1(10, 15, 8192) RGPU_DS1(11, 15, 9216)
		             RGPU_DS1(12, 15, 10240) RGPU_DS1(13, 15, 11264) "s_waitcnt lgkmcnt(0)"
		             : "=&v"(a[0]), "=&v"(a[1]), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3]), "=&v"(b[4]),
		               "=&v"(b[5]), "=&v"(b[6]), "=&v"(b[7]), "=&v"(b[8]), "=&v"(b[9]), "=&v"(b[10]), "=&v"(b[11])
		             : "v"(ab), "v"(bb)
		             : "memory");
	} else if constexpr (RT == 2 && CT == 8) {
		asm volatile(RGPU_DS1(0, 10, 0) RGPU_DS1(1, 10, 1024) RGPU_DS1(2, 11, 0) RGPU_DS1(3, 11, 1024)
		             RGPU_DS1(4, 11, 2048) RGPU_DS1(5, 11, 3072) RGPU_DS1(6, 11, 4096) RGPU_DS1(7, 11, 5120)
		             RGPU_DS1(8, 11, 6144) RGPU_DS1(9, 11, 7168) "s_waitcnt lgkmcnt(0)"
		             : "=&v"(a[0]), "=&v"(a[1]), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]), "=&v"(b[3]), "=&v"(b[4]),
		               "=&v"(b[5]), "=&v"(b[6]), "=&v"(b[7])
		             : "v"(ab), "v"(bb)
		             : "memory");
	} else if constexpr (RT == 4 && CT == 6) {
		asm volatile(RGPU_DS1(0, 10, 0) RGPU_DS1(1, 10, 1024) RGPU_DS1(2, 10, 2048) RGPU_DS1(3, 10, 3072)
		             RGPU_DS1(4, 11, 0) RGPU_DS1(5, 11, 1024) RGPU_DS1(6, 11, 2048) RGPU_DS1(7, 11, 3072)
		             RGPU_DS1(8, 11, 4096) RGPU_DS1(9, 11, 5120) "s_waitcnt lgkmcnt(0)"
		             : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]),
		               "=&v"(b[3]), "=&v"(b[4]), "=&v"(b[5])
		             : "v"(ab), "v"(bb)
		             : "memory");
	} else if constexpr (RT == 4 && CT == 4) {
		asm volatile(RGPU_DS1(0, 8, 0) RGPU_DS1(1, 8, 1024) RGPU_DS1(2, 8, 2048) RGPU_DS1(3, 8, 3072)
		             RGPU_DS1(4, 9, 0) RGPU_DS1(5, 9, 1024) RGPU_DS1(6, 9, 2048) RGPU_DS1(7, 9, 3072)
		             "s_waitcnt lgkmcnt(0)"
		             : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(b[0]), "=&v"(b[1]), "=&v"(b[2]),
		               "=&v"(b[3])
		             : "v"(ab), "v"(bb)
		             : "memory");
	} else {
		static_assert(RT < 0, "no slot reader for this tile");
	}
}
#undef RGPU_DS1

template <typename E, int NCT, int RT, int WC>
__global__ __launch_bounds__(512) void k_gemm_dma(const E *__restrict__ A, const E *__restrict__ XT,
                                                  float *__restrict__ part, int ld, int rp, int kchunk)
{
	typedef typename VecOf<E>::type V;
	constexpr int NS = 5, W = 8, WR = W / WC, CT = NCT / WC;
	constexpr int SLOT = (WR * RT + NCT) * 64;  // fragments (16 bytes) per ring slot
	// DMAs per wave and k-block: RT / WC of its row group's A fragments, and
	// BW of the B fragments, one more on waves w < BX
	constexpr int AW = RT / WC, BW = NCT / W, BX = NCT % W;
	static_assert(NCT == 8 || NCT == 12, "8 or 12 column tiles");
	static_assert(WR * RT == 16 && AW * WC == RT && CT * WC == NCT, "256 rows per block, whole splits");
	__shared__ V ring[NS * SLOT];
	const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int wr = w % WR, wc = w / WR;  // this wave's row group and column group
	const int rb0 = (blockIdx.x * WR + wr) * RT;
	// waves 4-7 (the second wave on each SIMD) run half a k-block behind:
	// their MFMAs on the previous k-block overlap the first four waves' LDS
	// reads, and their reads the others' MFMAs
	const bool late = w >= 4;
	const int s = blockIdx.y, kb0 = s * (kchunk >> 5), kb1 = kb0 + (kchunk >> 5);
	const int nkb = ld >> 5;
	const V *Ap = (const V *)A + lane, *Bp = (const V *)XT + lane;
	const bool extra = w < BX;
	const int c0 = w * BW + (extra ? w : BX);  // the first B fragment this wave loads
	f4 acc[RT][CT];
#pragma unroll
	for (int r = 0; r < RT; r++)
#pragma unroll
		for (int c = 0; c < CT; c++) acc[r][c] = f4{0.f, 0.f, 0.f, 0.f};
	auto issue = [&](int kb, int slot) {
		const int k = min(kb, kb1 - 1);
		V *base = ring + slot * SLOT;
		// A streams once: non-temporal (0.389 -> 0.364 ms at 192 columns);
		// B is read by every block and stays in L2
#pragma unroll
		for (int r = wc * AW; r < (wc + 1) * AW; r++)
			__builtin_amdgcn_global_load_lds((const void *)(Ap + ((size_t)(rb0 + r) * nkb + k) * 64),
			                                 (__attribute__((address_space(3))) void *)(base + (wr * RT + r) * 64), 16, 0,
			                                 kCpolNT);
#pragma unroll
		for (int m = 0; m < BW; m++)
			__builtin_amdgcn_global_load_lds((const void *)(Bp + ((size_t)(c0 + m) * nkb + k) * 64),
			                                 (__attribute__((address_space(3))) void *)(base + (WR * RT + c0 + m) * 64), 16, 0, 0);
		if (BX && extra)
			__builtin_amdgcn_global_load_lds((const void *)(Bp + ((size_t)(c0 + BW) * nkb + k) * 64),
			                                 (__attribute__((address_space(3))) void *)(base + (WR * RT + c0 + BW) * 64), 16, 0, 0);
	};
	const unsigned lbase = (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)ring + lane * 16;
	for (int i = 0; i < NS - 1; i++) issue(kb0 + i, i);
	int slot = 0;
	auto mma = [&](const V (&a)[RT], const V (&b)[CT]) {
#pragma unroll
		for (int r = 0; r < RT; r++)
#pragma unroll
			for (int c = 0; c < CT; c++) acc[r][c] = mfma(a[r], b[c], acc[r][c]);
	};
	// one k-block: its DMAs waited for, the barrier, the refill, then the
	// wave's own reads and MFMAs (body)
	auto step = [&](int kb, auto body) {
		// this k-block's DMAs: NS - 2 k-blocks' DMAs were issued after them
		constexpr int D = AW + BW;
		if (BX && extra) wait_vmcnt<(NS - 2) * (D + 1)>();
		else wait_vmcnt<(NS - 2) * D>();
		__builtin_amdgcn_s_barrier();
		// every wave is past its reads of the previous trip's slot: refill it
		issue(kb + NS - 1, slot == 0 ? NS - 1 : slot - 1);
		body(lbase + (unsigned)(slot * SLOT * 16 + wr * RT * 1024),
		     lbase + (unsigned)(slot * SLOT * 16 + (WR * RT + wc * CT) * 1024));
		slot = slot == NS - 1 ? 0 : slot + 1;
	};
	if (!late) {
		for (int kb = kb0; kb < kb1; kb++)
			step(kb, [&](unsigned ab, unsigned bb) {
				V a[RT], b[CT];
				read_slot<RT, CT>(a, b, ab, bb);
				mma(a, b);
			});
	} else {
		// the previous k-block's MFMAs, then this one's reads, into the
		// other of two fragment sets: no read overwrites an operand of an
		// MFMA issued in the same trip
		V a0[RT], b0[CT], a1[RT], b1[CT];
		step(kb0, [&](unsigned ab, unsigned bb) { read_slot<RT, CT>(a0, b0, ab, bb); });
		for (int kb = kb0 + 1; kb < kb1; kb += 2) {
			step(kb, [&](unsigned ab, unsigned bb) {
				mma(a0, b0);
				read_slot<RT, CT>(a1, b1, ab, bb);
			});
			if (kb + 1 < kb1)
				step(kb + 1, [&](unsigned ab, unsigned bb) {
					mma(a1, b1);
					read_slot<RT, CT>(a0, b0, ab, bb);
				});
		}
		if ((kb1 - kb0) & 1) mma(a0, b0);  // the last k-block went to set 0
		else mma(a1, b1);
	}
	asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no DMA may outlive the block's LDS
	const int lr = lane & 15;
#pragma unroll
	for (int r = 0; r < RT; r++)
#pragma unroll
		for (int c = 0; c < CT; c++)
#pragma unroll
			for (int j = 0; j < 4; j++) {
				const int row = (rb0 + r) * 16 + (lane >> 4) * 4 + j;
				part[((size_t)s * ld + row) * rp + (wc * CT + c) * 16 + lr] = acc[r][c][j];
			}
}

// The element-wise kernels take R rows of one column per thread, columns across
// the lanes (unit u -> rows [i, i + R) of column c).  R = 8 from 2^19 elements
// up: the row-major arrays are read a line at a time, and a column's rows, 16
// bytes of a fragment (frag_index) or 64 of the FP64 iterate, are one access
// where an element per thread touches as many lines as lanes.  Below, one: there
// it is threads that are short.  us at (n, columns), one row and eight: k_resid
// (1000, 6) 5.5, 7.8; (4000, 96) 9.8, 9.4; (6000, 192) 27.5, 22.6; k_finish
// (1000, 96) 4.1, 4.8; (4000, 96) 4.8, 4.8; (6000, 192) 14.8, 10.3; k_scale
// (20000, 3) 2.9, 4.3; (4000, 96) 3.6, 5.2; (6000, 192) 7.2, 6.1.
constexpr size_t kWide = (size_t)1 << 19;
constexpr size_t row_units(int R, int n, int nrhs) { return (size_t)((n + R - 1) / R) * nrhs; }

// The sweep's second half after k_gemm_dma: its split-K partials summed in
// order.  Bound by the partials' and vectors' traffic: n = 7777, 192 columns, 8
// partials, 17.2 us with one row, 11.8 (5.3 TB/s) with eight.
template <typename E, int R>
__global__ __launch_bounds__(kB) void k_finish(const float *part, int S, int ld, int rp, SweepOut<E> o)
{
	const size_t u = blockIdx.x * (size_t)kB + threadIdx.x;
	if (u >= row_units(R, o.n, o.nrhs)) return;
	const int i = (int)(u / o.nrhs) * R, c = (int)(u % o.nrhs), m = min(R, o.n - i);
	float y[R] = {};
	const float *p = part + (size_t)i * rp + c;  // whole row groups: ld is a multiple of 256
	for (int s = 0; s < S; s++)
#pragma unroll
		for (int r = 0; r < R; r++) y[r] += p[((size_t)s * ld + r) * rp];
	E x[R];
#pragma unroll
	for (int r = 0; r < R; r++) x[r] = r < m ? o.value(i + r, c, ld, y[r]) : (E)0.f;
	if (!o.y) put_frag<R>(o.XTn, c, i, ld, x);
}

// Split-K partials part[s][row][col] (FP64) of F X, summed in a fixed order
// by k_resid, on the FP64 MFMA (v_mfma_f64_16x16x4_f64: lane l supplies
// A[l%16][l/16] and B[l/16][l%16], receives D[l/16 + 4*j][l%16], j = 0..3 --
// rows interleaved, unlike the 16-bit MFMAs).  A block is W waves of 16 RT rows
// each over the same 16 CT columns, whose 32 k per step they stage in LDS (two
// buffers, columns 34 doubles apart: the 16-byte reads of 16 columns fall on all
// 64 banks; 3.5 conflict cycles an instruction are left); a lane loads 8 consecutive F entries of its row per step
// (converted exactly to FP64), the next step's on their way, and step s pairs
// k = kk + 8*(l/16) + s in both operands, so every k is summed once.
// Bound by the FP64 matrix units (busy 0.81 of the cycles at n = 7777, 192 columns;
// 73 TFLOP/s in a large library product); with
// each wave reading its own X from L2 it was that traffic (12 TB/s).  us at n =
// 7936, 16, 32, 64, 192 columns: 67, 103, 172, 486 -> 45, 75, 131, 382 (63
// TFLOP/s); n = 1024, 16 and 64: 9.2, 13.2 -> 4.6, 9.2; n = 16384, 192: 1850 ->
// 1513 (68 TFLOP/s).
template <int RT, int CT, int W>
__global__ __launch_bounds__(W * 64) void k_fx64m(const float *__restrict__ F, const double *__restrict__ xT,
                                                  double *__restrict__ part, int ld, int rp, int kchunk)
{
	typedef double d4 __attribute__((ext_vector_type(4)));
	typedef double dv2 __attribute__((ext_vector_type(2)));
	typedef float fv4 __attribute__((ext_vector_type(4)));
	constexpr int PAD = 34, NL = CT * 16 * 16 / (W * 64);  // 16-byte loads of X per thread and step
	static_assert(NL * W * 64 == CT * 16 * 16, "whole loads");
	__shared__ double bs[2][CT * 16 * PAD];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, g8 = (lane >> 4) * 8;
	const int rb0 = (blockIdx.x * W + w) * RT, cb0 = blockIdx.y * CT;
	const int k0 = blockIdx.z * kchunk, k1 = k0 + kchunk;
	const float *Fr[RT];
#pragma unroll
	for (int r = 0; r < RT; r++) Fr[r] = F + (size_t)((rb0 + r) * 16 + lr) * ld + g8;
	d4 acc[RT][CT];
#pragma unroll
	for (int r = 0; r < RT; r++)
#pragma unroll
		for (int c = 0; c < CT; c++) acc[r][c] = d4{0.0, 0.0, 0.0, 0.0};
	fv4 a[RT][2], an[RT][2];
	dv2 sb[NL];
	auto load_x = [&](int kk) {
#pragma unroll
		for (int i = 0; i < NL; i++) {
			const int e = threadIdx.x + i * W * 64;  // 16 loads per column
			sb[i] = *(const dv2 *)(xT + (size_t)(cb0 * 16 + e / 16) * ld + kk + 2 * (e % 16));
		}
	};
	auto store_x = [&](int p) {
#pragma unroll
		for (int i = 0; i < NL; i++) {
			const int e = threadIdx.x + i * W * 64;
			*(dv2 *)(&bs[p][(e / 16) * PAD + 2 * (e % 16)]) = sb[i];
		}
	};
	auto load_f = [&](fv4 (&x)[RT][2], int kk) {
#pragma unroll
		for (int r = 0; r < RT; r++) {
			x[r][0] = ((const fv4 *)(Fr[r] + kk))[0];
			x[r][1] = ((const fv4 *)(Fr[r] + kk))[1];
		}
	};
	load_x(k0);
	load_f(a, k0);
	store_x(0);
	__syncthreads();
	int p = 0;
	for (int kk = k0; kk < k1; kk += 32) {
		const int kn = kk + 32 < k1 ? kk + 32 : kk;  // the last step's loads are not used
		load_x(kn);
		load_f(an, kn);
#pragma unroll
		for (int h = 0; h < 4; h++) {
			dv2 b[CT];
#pragma unroll
			for (int c = 0; c < CT; c++) b[c] = *(const dv2 *)(&bs[p][(c * 16 + lr) * PAD + g8 + 2 * h]);
#pragma unroll
			for (int u = 0; u < 2; u++)
#pragma unroll
				for (int r = 0; r < RT; r++) {
					const double f = (double)a[r][h >> 1][(h & 1) * 2 + u];
#pragma unroll
					for (int c = 0; c < CT; c++) acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(f, b[c][u], acc[r][c], 0, 0, 0);
				}
		}
		store_x(p ^ 1);  // its readers are past the previous step's barrier
		__syncthreads();
		p ^= 1;
#pragma unroll
		for (int r = 0; r < RT; r++) {
			a[r][0] = an[r][0];
			a[r][1] = an[r][1];
		}
	}
	double *P = part + (size_t)blockIdx.z * ld * rp;
#pragma unroll
	for (int r = 0; r < RT; r++)
#pragma unroll
		for (int c = 0; c < CT; c++)
#pragma unroll
			for (int j = 0; j < 4; j++)
				P[(size_t)((rb0 + r) * 16 + (lane >> 4) + 4 * j) * rp + (cb0 + c) * 16 + lr] = acc[r][c][j];
}

template <int NC, int KS>
__global__ __launch_bounds__(kB) void k_fx64v(const float *__restrict__ F, const double *__restrict__ wT, int ld, int n,
                                              const double *xT, const double *base, const double *rho, double *out,
                                              double *blk)
{
	__shared__ FxShared<NC, KS> sh;
	fx64_rows<NC, KS>(F, wT, ld, n, blockIdx.x, sh, xT, base, rho, out, blk + 2 * blockIdx.x);
}

// out[i][c] = base[i][c] + rho[i][c] * y - xT[c][i], y = the split-K sum of
// part (FP64, fixed order); base, rho and xT may be null (0, 1 and 0).  Per
// block: sum of squares and max |out|.
template <int R>
__global__ __launch_bounds__(kB) void k_resid(const double *part, int S, int ld, int rp, int n, int nrhs,
                                              const double *xT, const double *base, const double *rho, double *out,
                                              double *blk)
{
	const size_t u = blockIdx.x * (size_t)kB + threadIdx.x;
	double ss = 0.0, mx = 0.0;
	if (u < row_units(R, n, nrhs)) {
		const int i = (int)(u / nrhs) * R, c = (int)(u % nrhs), m = min(R, n - i);
		double y[R] = {}, x[R] = {};
		const double *p = part + (size_t)i * rp + c;
		for (int q = 0; q < S; q++)
#pragma unroll
			for (int r = 0; r < R; r++) y[r] += p[((size_t)q * ld + r) * rp];
		if (xT)
#pragma unroll
			for (int r = 0; r < R; r++) x[r] = xT[(size_t)c * ld + i + r];
#pragma unroll
		for (int r = 0; r < R; r++) {
			if (r >= m) break;
			const size_t t = (size_t)(i + r) * nrhs + c;
			const double v = (base ? base[t] : 0.0) + (rho ? rho[t] : 1.0) * y[r] - x[r];
			out[t] = v;
			ss += v * v;
			mx = fmax(mx, fabs(v));
		}
	}
	for (int off = 32; off > 0; off >>= 1) {
		ss += __shfl_xor(ss, off);
		mx = fmax(mx, __shfl_xor(mx, off));
	}
	__shared__ double r[8];
	if ((threadIdx.x & 63) == 0) {
		r[2 * (threadIdx.x >> 6)] = ss;
		r[2 * (threadIdx.x >> 6) + 1] = mx;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		blk[2 * blockIdx.x] = r[0] + r[2] + r[4] + r[6];
		blk[2 * blockIdx.x + 1] = fmax(fmax(r[1], r[3]), fmax(r[5], r[7]));
	}
}

// r32 = r64 / s; XT <- r32 (times rho_in, if given) in fragment order
template <typename E, int R>
__global__ __launch_bounds__(kB) void k_scale(const double *r64, double inv_s, int n, int nrhs, int ld, float *r32, E *XT,
                                              const float *rho_in)
{
	const size_t u = blockIdx.x * (size_t)kB + threadIdx.x;
	if (u >= row_units(R, n, nrhs)) return;
	const int i = (int)(u / nrhs) * R, c = (int)(u % nrhs), m = min(R, n - i);
	E x[R];
#pragma unroll
	for (int r = 0; r < R; r++) {
		const size_t t = (size_t)min(i + r, n - 1) * nrhs + c;
		const float v = (float)(r64[t] * inv_s);
		if (r < m) r32[t] = v;
		x[r] = r < m ? (E)(rho_in ? rho_in[t] * v : v) : (E)0.f;
	}
	put_frag<R>(XT, c, i, ld, x);
}

// rho32 <- rho and per block (grid-stride): sum of squares and max of |E|, the
// power sum_i area_i E_i; rho and E go to rho64 and E64 where those are others
constexpr int kStatBlocks = 1024;
__global__ __launch_bounds__(kB) void k_prep(const double *rho, const double *E, const float *area, unsigned total,
                                             unsigned nrhs, float *rho32, double *stat, double *rho64, double *E64)
{
	double ss = 0.0, mx = 0.0, pw = 0.0;
	for (unsigned t = blockIdx.x * kB + threadIdx.x; t < total; t += gridDim.x * kB) {
		const double e = E[t], p = rho[t];
		rho32[t] = (float)p;
		if (rho64 != rho) {
			rho64[t] = p;
			E64[t] = e;
		}
		ss += e * e;
		mx = fmax(mx, fabs(e));
		pw += (double)area[t / nrhs] * e;
	}
	for (int off = 32; off > 0; off >>= 1) {
		ss += __shfl_xor(ss, off);
		mx = fmax(mx, __shfl_xor(mx, off));
		pw += __shfl_xor(pw, off);
	}
	__shared__ double r[12];
	if ((threadIdx.x & 63) == 0) {
		r[3 * (threadIdx.x >> 6)] = ss;
		r[3 * (threadIdx.x >> 6) + 1] = mx;
		r[3 * (threadIdx.x >> 6) + 2] = pw;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		stat[3 * blockIdx.x] = r[0] + r[3] + r[6] + r[9];
		stat[3 * blockIdx.x + 1] = fmax(fmax(r[1], r[4]), fmax(r[7], r[10]));
		stat[3 * blockIdx.x + 2] = r[2] + r[5] + r[8] + r[11];
	}
}

// xT[c][i] = in[i][c], and out[i][c] = (mul ? mul[i][c] : 1) * xT[c][i] with,
// per block (pw given), the power sum_i area_i xT[.][i]: 64 rows by up to 64
// columns a block, turned through LDS so that both sides are contiguous
constexpr int kTurn = 64;
__global__ __launch_bounds__(kB) void k_cols(const double *in, int ld, int n, int nrhs, double *xT)
{
	__shared__ double tile[kTurn][kTurn + 1];
	const int i0 = blockIdx.x * kTurn, c0 = blockIdx.y * kTurn, nc = min(kTurn, nrhs - c0), ni = min(kTurn, n - i0);
	for (int e = threadIdx.x; e < ni * nc; e += kB) tile[e / nc][e % nc] = in[(size_t)(i0 + e / nc) * nrhs + c0 + e % nc];
	__syncthreads();
	for (int e = threadIdx.x; e < kTurn * nc; e += kB)
		if (e % kTurn < ni) xT[(size_t)(c0 + e / kTurn) * ld + i0 + e % kTurn] = tile[e % kTurn][e / kTurn];
}
__global__ __launch_bounds__(kB) void k_rows(const double *xT, int ld, int n, int nrhs, const double *mul, double *out,
                                             const float *area, double *pw)
{
	__shared__ double tile[kTurn][kTurn + 1];
	const int i0 = blockIdx.x * kTurn, c0 = blockIdx.y * kTurn, nc = min(kTurn, nrhs - c0), ni = min(kTurn, n - i0);
	double p = 0.0;
	for (int e = threadIdx.x; e < kTurn * nc; e += kB)
		if (e % kTurn < ni) {
			const double x = xT[(size_t)(c0 + e / kTurn) * ld + i0 + e % kTurn];
			tile[e % kTurn][e / kTurn] = x;
			if (pw) p += (double)area[i0 + e % kTurn] * x;
		}
	__syncthreads();
	for (int e = threadIdx.x; e < ni * nc; e += kB) {
		const size_t t = (size_t)(i0 + e / nc) * nrhs + c0 + e % nc;
		const double x = tile[e / nc][e % nc];
		out[t] = mul ? x * mul[t] : x;
	}
	if (!pw) return;
	for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off);
	__shared__ double r[4];
	if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = p;
	__syncthreads();
	if (threadIdx.x == 0) pw[blockIdx.y * gridDim.x + blockIdx.x] = r[0] + r[1] + r[2] + r[3];
}
dim3 turn_grid(int n, int nrhs) { return dim3((n + kTurn - 1) / kTurn, (nrhs + kTurn - 1) / kTurn); }

// per block: sum (x - ref)^2 and sum ref^2 (x transposed [c][ld] or row-major)
__global__ void k_err(const double *x, int transposed, int ld, const double *ref, int n, int nrhs, double *blk)
{
	const size_t total = (size_t)n * nrhs;
	double a = 0.0, b = 0.0;
	for (size_t t = blockIdx.x * (size_t)kB + threadIdx.x; t < total; t += (size_t)gridDim.x * kB) {
		const double xv = transposed ? x[(size_t)(t % nrhs) * ld + t / nrhs] : x[t];
		const double e = xv - ref[t];
		a += e * e;
		b += ref[t] * ref[t];
	}
	for (int off = 32; off > 0; off >>= 1) {
		a += __shfl_xor(a, off);
		b += __shfl_xor(b, off);
	}
	__shared__ double r[8];
	if ((threadIdx.x & 63) == 0) {
		r[2 * (threadIdx.x >> 6)] = a;
		r[2 * (threadIdx.x >> 6) + 1] = b;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		blk[2 * blockIdx.x] = r[0] + r[2] + r[4] + r[6];
		blk[2 * blockIdx.x + 1] = r[1] + r[3] + r[5] + r[7];
	}
}

// ---- plain progressive shooting (FP32) --------------------------------------
// One launch per shot, no atomics and no device-wide fences.  Launch k reads
// the per-block records of launch k-1 (each: the block's largest unshot-power
// key, area_i * sum_c dB_i[c] with ties to the lowest index, and that patch's
// dB row), reduces them to the source j and its dB_j, adds
// rho_i F_ij dB_j to B_i and dB_i for every patch i (the source's own dB
// restarting from 0), and writes its own records for launch k+1.  Records are
// double-buffered by shot parity.  A zero best key means nothing is left to
// shoot: the launch only passes the zero on.
constexpr int kMaxShootRhs = 16;
struct ShotRec {
	unsigned long long key;
	float dB[kMaxShootRhs];
	float pad[2];
};

__device__ __forceinline__ unsigned long long power_key(float p, int j)
{
	// p > 0 here, so its bits order as the value
	return ((unsigned long long)__float_as_uint(p) << 32) | (0xffffffffu - (uint32_t)j);
}

__device__ __forceinline__ unsigned long long wave_max(unsigned long long key)
{
	for (int off = 32; off > 0; off >>= 1) {
		const unsigned long long o = __shfl_xor(key, off);
		key = o > key ? o : key;
	}
	return key;
}

// block maximum of key; the thread holding it writes its dB row to rec
__device__ __forceinline__ void block_record(unsigned long long key, const float *row, int nrhs, ShotRec *rec)
{
	__shared__ unsigned long long wk[4];
	const unsigned long long wm = wave_max(key);
	if ((threadIdx.x & 63) == 0) wk[threadIdx.x >> 6] = wm;
	__syncthreads();
	unsigned long long m = wk[0];
	for (int w = 1; w < 4; w++) m = wk[w] > m ? wk[w] : m;
	if (threadIdx.x == 0) rec->key = m;
	if (m != 0 && key == m)  // keys are unique (the index is in them)
		for (int c = 0; c < nrhs; c++) rec->dB[c] = row[c];
}

// The same shots in one launch, where one block's registers hold the system:
// 1024 threads, R patches each (i = thread + 1024 r), C >= nrhs columns, with
// R (3 C + 3) <= kOneState values a thread (radiosity, unshot, reflectance, area
// and two matrix columns).  Per shot the patches' keys are reduced over the wave's
// lanes (DPP), the wave's largest and its dB row meet the others' in LDS (two
// sets by parity: one barrier a shot), and every wave takes the block's
// largest from there.  The runner-up's column is loaded while the source's is
// on its way: mostly it is the next source.
// Bound by one CU's VALU issue, 0.85 of its cycles at n = 4000 with 3 columns (191
// instructions a wave and shot) and 0.88 at 12000 with 1, and by the dependent
// chain (a latency where the guess fails, two reductions, a barrier), whose share
// is larger in small systems (issue 0.61 at n = 500, 0.69 at 2000) and where the
// columns no longer stay in cache (0.72 at 8000).  us per shot for 3 columns, a
// launch per shot -> now: n = 500 4.00 -> 0.85, 2000 4.23 -> 1.16, 4000 4.32 ->
// 1.55, 8000 4.41 -> 2.87; 1 column, n = 12000 3.71 -> 2.25.  16 patches a thread
// (1 column, n = 16000) spill: 4.82 against 3.74, so twelve is the most.
constexpr int kOneThreads = 1024;
constexpr int kOneState = 100;

// maximum over the wave (row_shr 1, 2, 4, 8, then row_bcast 15 and 31; lanes
// without a source give 0), in every lane
__device__ __forceinline__ uint32_t row_max(uint32_t x)
{
	x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x111, 0xf, 0xf, false));
	x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x112, 0xf, 0xf, false));
	x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x114, 0xf, 0xf, false));
	x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x118, 0xf, 0xf, false));
	return x;  // lane 15 of each row of 16 holds the row's
}
__device__ __forceinline__ uint32_t lane_max(uint32_t x)
{
	x = row_max(x);
	x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x142, 0xa, 0xf, false));
	x = max(x, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x143, 0xc, 0xf, false));
	return (uint32_t)__builtin_amdgcn_readlane((int)x, 63);
}
// the lane of `who` with the lowest idx (who != 0)
__device__ __forceinline__ int lowest(unsigned long long who, int idx)
{
	int l = __ffsll((long long)who) - 1;
	int best = __builtin_amdgcn_readlane(idx, l);
	for (who &= who - 1; who; who &= who - 1) {  // ties only
		const int m = __ffsll((long long)who) - 1, i = __builtin_amdgcn_readlane(idx, m);
		if (i < best) {
			best = i;
			l = m;
		}
	}
	return l;
}

template <int R, int C>
__global__ __launch_bounds__(kOneThreads) void k_lshoot_one(const float *__restrict__ Ft, int ld, const float *rho,
                                                            const float *area, float *B, float *dB, int n, int nrhs,
                                                            int shots, int *done)
{
	constexpr int NW = kOneThreads / 64;
	static_assert(NW == 16, "one row of 16 lanes reduces the waves' records");
	// per parity and wave: its largest power, that patch, its dB row; the power
	// and patch of its second largest
	__shared__ uint32_t pw[2][NW], pw2[2][NW];
	__shared__ int ix[2][NW], ix2[2][NW];
	__shared__ float row[2][NW][C];
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	float b[R][C], d[R][C], rh[R][C], ar[R], f[R], g[R];
#pragma unroll
	for (int r = 0; r < R; r++) {
		const int i = threadIdx.x + kOneThreads * r;
		ar[r] = i < n ? area[i] : 0.f;
#pragma unroll
		for (int c = 0; c < C; c++) {
			const bool in = i < n && c < nrhs;
			const size_t t = (size_t)i * nrhs + c;
			b[r][c] = in ? B[t] : 0.f;
			d[r][c] = in ? dB[t] : 0.f;
			rh[r][c] = in ? rho[t] : 0.f;
		}
		g[r] = 0.f;
	}
	int guess = -1;  // the patch whose column g holds
	int k = 0;
	for (; k < shots; k++) {
		const int q = k & 1;
		// this thread's two largest (the lower patch on ties)
		uint32_t p1 = 0, p2 = 0;
		int i1 = 0, i2 = 0, r1 = 0;
#pragma unroll
		for (int r = 0; r < R; r++) {
			float p = 0.f;
#pragma unroll
			for (int c = 0; c < C; c++) p += d[r][c];
			p *= ar[r];
			const uint32_t u = p > 0.f ? __float_as_uint(p) : 0u;
			const int i = threadIdx.x + kOneThreads * r;
			if (u > p1) {
				p2 = p1, i2 = i1;
				p1 = u, i1 = i, r1 = r;
			} else if (u > p2) {
				p2 = u, i2 = i;
			}
		}
		// the wave's: its winner's lane also gives the runner-up up for the rest
		const uint32_t wm = lane_max(p1);
		const int wl = wm ? lowest(__ballot(p1 == wm), i1) : 0;
		const uint32_t s1 = lane == wl ? p2 : p1;
		const int si = lane == wl ? i2 : i1;
		const uint32_t wm2 = lane_max(s1);
		const int wl2 = wm2 ? __ffsll((long long)__ballot(s1 == wm2)) - 1 : 0;
		if (lane == wl) {
			pw[q][w] = wm;
			ix[q][w] = i1;
#pragma unroll
			for (int r = 0; r < R; r++)
				if (r == r1)
#pragma unroll
					for (int c = 0; c < C; c++) row[q][w][c] = d[r][c];
		}
		if (lane == wl2) {
			pw2[q][w] = wm2;
			ix2[q][w] = si;
		}
		__syncthreads();
		// the block's, in every wave
		const uint32_t bp = pw[q][lane & 15], bp2 = pw2[q][lane & 15];
		const int bi = ix[q][lane & 15], bi2 = ix2[q][lane & 15];
		const uint32_t best = (uint32_t)__builtin_amdgcn_readlane((int)row_max(bp), 15);
		if (best == 0) break;  // nothing left to shoot
		const int ws = lowest(__ballot(bp == best) & 0xffffull, bi);
		const int j = __builtin_amdgcn_readlane(bi, ws);
		const float *col = Ft + (size_t)j * ld;
		if (j != guess) {
#pragma unroll
			for (int r = 0; r < R; r++) f[r] = col[min((int)threadIdx.x + kOneThreads * r, n - 1)];
		} else {
#pragma unroll
			for (int r = 0; r < R; r++) f[r] = g[r];
		}
		// the runner-up: the largest of the other waves' first and this one's second
		const uint32_t t1 = (lane & 15) == ws ? bp2 : bp;
		const int ti = (lane & 15) == ws ? bi2 : bi;
		const uint32_t second = (uint32_t)__builtin_amdgcn_readlane((int)row_max(t1), 15);
		guess = -1;
		if (second) {
			guess = __builtin_amdgcn_readlane(ti, __ffsll((long long)(__ballot(t1 == second) & 0xffffull)) - 1);
			const float *c2 = Ft + (size_t)guess * ld;
#pragma unroll
			for (int r = 0; r < R; r++) g[r] = c2[min((int)threadIdx.x + kOneThreads * r, n - 1)];
		}
		float src[C];
#pragma unroll
		for (int c = 0; c < C; c++) src[c] = row[q][ws][c];
#pragma unroll
		for (int r = 0; r < R; r++) {
			const bool self = (int)threadIdx.x + kOneThreads * r == j;
#pragma unroll
			for (int c = 0; c < C; c++) {
				const float v = rh[r][c] * f[r] * src[c];
				b[r][c] += v;
				d[r][c] = (self ? 0.f : d[r][c]) + v;
			}
		}
	}
#pragma unroll
	for (int r = 0; r < R; r++) {
		const int i = threadIdx.x + kOneThreads * r;
#pragma unroll
		for (int c = 0; c < C; c++)
			if (i < n && c < nrhs) {
				B[(size_t)i * nrhs + c] = b[r][c];
				dB[(size_t)i * nrhs + c] = d[r][c];
			}
	}
	if (threadIdx.x == 0) *done += k;
}

// launches k_lshoot_one for the system, or returns false where it is too large
// for one block
bool launch_shoot_one(const float *Ft, int ld, const float *rho, const float *area, float *B, float *dB, int n,
                      int nrhs, int shots, int *done, hipStream_t st)
{
	const int r = (n + kOneThreads - 1) / kOneThreads;
	bool ok = false;
	auto go = [&](auto rc, auto cc) {
		constexpr int R = decltype(rc)::value, C = decltype(cc)::value;
		if constexpr (R * (3 * C + 3) <= kOneState) {
			if (ok || r > R || nrhs > C) return;
			hipLaunchKernelGGL((k_lshoot_one<R, C>), dim3(1), dim3(kOneThreads), 0, st, Ft, ld, rho, area, B, dB, n, nrhs,
			                   shots, done);
			ok = true;
		}
	};
	auto rows = [&](auto cc) {
		go(std::integral_constant<int, 1>{}, cc);
		go(std::integral_constant<int, 2>{}, cc);
		go(std::integral_constant<int, 4>{}, cc);
		go(std::integral_constant<int, 6>{}, cc);
		go(std::integral_constant<int, 8>{}, cc);
		go(std::integral_constant<int, 12>{}, cc);
	};
	if (nrhs <= 1) rows(std::integral_constant<int, 1>{});
	else if (nrhs <= 3) rows(std::integral_constant<int, 3>{});
	else if (nrhs <= 6) rows(std::integral_constant<int, 6>{});
	else if (nrhs <= 12) rows(std::integral_constant<int, 12>{});
	else rows(std::integral_constant<int, 16>{});
	return ok;
}

// records of the initial dB (launch 0's input)
__global__ __launch_bounds__(kB) void k_lsel(const float *dB, const float *area, int n, int nrhs, ShotRec *rout)
{
	const int i = blockIdx.x * kB + threadIdx.x;
	unsigned long long key = 0;
	float row[kMaxShootRhs];
	if (i < n) {
		float p = 0.f;
		for (int c = 0; c < nrhs; c++) {
			row[c] = dB[(size_t)i * nrhs + c];
			p += row[c];
		}
		p *= area[i];
		if (p > 0.f) key = power_key(p, i);
	}
	block_record(key, row, nrhs, rout + blockIdx.x);
}

__global__ __launch_bounds__(kB) void k_lshoot(const float *__restrict__ Ft, int ld, const float *rho, const float *area,
                                               float *B, float *dB, int n, int nrhs, const ShotRec *rin,
                                               ShotRec *rout, int *shots)
{
	__shared__ unsigned long long wk[4];
	__shared__ int sb;
	__shared__ float src[kMaxShootRhs];
	// the previous launch's records -> source
	unsigned long long k = 0;
	for (int b = threadIdx.x; b < (int)gridDim.x; b += kB) {
		const unsigned long long o = rin[b].key;
		k = o > k ? o : k;
	}
	const unsigned long long wm = wave_max(k);
	if ((threadIdx.x & 63) == 0) wk[threadIdx.x >> 6] = wm;
	__syncthreads();
	unsigned long long best = wk[0];
	for (int w = 1; w < 4; w++) best = wk[w] > best ? wk[w] : best;
	if (best == 0) {  // nothing left to shoot (uniform over the grid)
		if (threadIdx.x == 0) rout[blockIdx.x].key = 0;
		return;
	}
	for (int b = threadIdx.x; b < (int)gridDim.x; b += kB)
		if (rin[b].key == best) sb = b;
	__syncthreads();
	if (threadIdx.x < nrhs) src[threadIdx.x] = rin[sb].dB[threadIdx.x];
	__syncthreads();
	const int j = (int)(0xffffffffu - (uint32_t)best);
	const int i = blockIdx.x * kB + threadIdx.x;
	unsigned long long key = 0;
	float row[kMaxShootRhs];
	if (i < n) {
		const float f = Ft[(size_t)j * ld + i];
		float p = 0.f;
		for (int c = 0; c < nrhs; c++) {
			const size_t t = (size_t)i * nrhs + c;
			const float v = rho[t] * f * src[c];
			B[t] += v;
			const float nd = (i == j ? 0.f : dB[t]) + v;
			dB[t] = nd;
			row[c] = nd;
			p += nd;
		}
		p *= area[i];
		if (p > 0.f) key = power_key(p, i);
	}
	block_record(key, row, nrhs, rout + blockIdx.x);
	if (blockIdx.x == 0 && threadIdx.x == 0) *shots += 1;  // launches on one stream: no race
}

__global__ void k_transpose(const float *F, float *Ft, int ld)
{
	__shared__ float tile[32][33];
	const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
	const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: 32 x 8
	for (int r = ty; r < 32; r += 8) tile[r][tx] = F[(size_t)(by + r) * ld + bx + tx];
	__syncthreads();
	for (int r = ty; r < 32; r += 8) Ft[(size_t)(bx + r) * ld + by + tx] = tile[tx][r];
}

const int kCT[] = {1, 2, 4, 8, 12};
int pick_ct(int nrhs)
{
	const int need = (nrhs + 15) / 16;
	for (int c : kCT)
		if (c >= need) return c;
	return -1;
}

// go(integral constant R, grid) for an element-wise kernel over n x nrhs
template <typename Go> void launch_rows(int n, int nrhs, Go go)
{
	auto grid = [&](int R) { return dim3((unsigned)((row_units(R, n, nrhs) + kB - 1) / kB)); };
	if ((size_t)n * nrhs >= kWide) go(std::integral_constant<int, 8>{}, grid(8));
	else go(std::integral_constant<int, 1>{}, grid(1));
}
template <typename E>
void launch_scale(const double *r64, double inv_s, int n, int nrhs, int ld, float *r32, E *XT, const float *rho_in,
                  hipStream_t st)
{
	launch_rows(n, nrhs, [&](auto r, dim3 g) {
		hipLaunchKernelGGL((k_scale<E, decltype(r)::value>), g, dim3(kB), 0, st, r64, inv_s, n, nrhs, ld, r32, XT, rho_in);
	});
}

// the wide kernels' tiles: split-K over blocks, partials in part
bool dma_tile(int rt, int ct) { return ct >= 8 && rt >= 2; }

// The sweep's tile for ct <= 4 where none was tuned or forced: the smallest
// row group whose blocks fit the 256 CUs in one round (16, 32, 64 rows a block
// with every wave on the same rows, or 128).  Of the twelve tiles, timed at 21
// sizes from 512 to 32768 rows, this one is the fastest or within 6 % of it
// (one column tile, us: n = 4096 (1, 8) 5.4, (2, 8) 6.2; 6144 (1, 8) 13.7, (2,
// 8) 12.5; 9216 (2, 8) 30.7, (4, 8) 24.7; four column tiles: 20224 (4, 8)
// 205.3, (4, 4) 197.6).  Past 16384 rows one column tile does better with more
// blocks of 32 rows (20224: 136.3 against 142.2).
// Wide (ct 8 and 12): up to 4096 rows and eight column tiles 16 rows a block as
// above; else k_gemm_dma's 256 rows, K split as often as the blocks still fit the
// CUs in one round (twelve column tiles below 1280 rows: four ways, as each
// partial is then a sixth of the work).  Of the twelve tiles at 17 sizes from 512
// to 20224 rows, both precisions, the fastest or within 5 % of it, with k_finish
// (us: eight column tiles, 4096 (1, 8) 16.9, (4, 8) 20.1; 5120 (1, 8) 36.6, (4, 8)
// 23.5; twelve, 7936 (2, 8) 44.4, (2, 4) 54.1; 10240 (2, 8) 78.2, (2, 4) 68.1;
// 20224 (2, 4) 222, (2, 2) 211).  Timing them on the first solve took 9 ms at
// 7777 rows.
void sweep_tile(int ct, int ld, int &rt, int &S)
{
	rt = ld <= 4096 ? 1 : ld <= 8192 ? 2 : 4;
	S = 8;
	if (ct > 4 && (ct > 8 || ld > 4096)) {
		rt = ct > 8 ? 2 : 4;
		while (S > 1 && ld / 256 * S > 256) S /= 2;
		if (ld < 1280) S = 4;
	} else if (ld > 16384) {
		rt = ct == 1 ? 2 : 4;
		S = ct == 1 ? 8 : 4;
	}
}

// One product with the tile (rt, S) and what follows it (o).  finish = false:
// the wide tiles' product only (for timing it alone).  ld is a multiple of 256,
// so rt 1, 2 and 4 and S 1, 2, 4 and 8 go with every size: k_sweep clamps its
// rows and k-blocks, and k_gemm_dma's 256 rows and S chunks of at least 32 k
// divide it.
template <typename E>
int launch_sweep(int rt, int ct, int S, const E *A, const E *XT, float *part, int ld, int rp, const SweepOut<E> &o,
                 hipStream_t st, bool finish = true)
{
	if (dma_tile(rt, ct)) {
		const dim3 grid(ld / 256, S), blk(512);
		const int kchunk = ld / S;
		if (rt == 2 && ct == 8) hipLaunchKernelGGL((k_gemm_dma<E, 8, 2, 1>), grid, blk, 0, st, A, XT, part, ld, rp, kchunk);
		else if (rt == 2 && ct == 12) hipLaunchKernelGGL((k_gemm_dma<E, 12, 2, 1>), grid, blk, 0, st, A, XT, part, ld, rp, kchunk);
		else if (rt == 4 && ct == 8) hipLaunchKernelGGL((k_gemm_dma<E, 8, 4, 2>), grid, blk, 0, st, A, XT, part, ld, rp, kchunk);
		else if (rt == 4 && ct == 12) hipLaunchKernelGGL((k_gemm_dma<E, 12, 4, 2>), grid, blk, 0, st, A, XT, part, ld, rp, kchunk);
		else return -1;
		if (finish)
			launch_rows(o.n, o.nrhs, [&](auto r, dim3 g) {
				hipLaunchKernelGGL((k_finish<E, decltype(r)::value>), g, dim3(kB), 0, st, part, S, ld, rp, o);
			});
		return 0;
	}
	const int wr = kSweepWaves / S * rt;  // row tiles per block
	const dim3 grid((ld / 16 + wr - 1) / wr), blk(kSweepWaves * 64);
	const bool cached = stays_cached((size_t)ld * ld);
#define G(R, C) \
	if (rt == R && ct == C) { \
		hipLaunchKernelGGL((k_sweep<E, R, C>), grid, blk, 0, st, A, XT, ld, S, cached, o); \
		return 0; \
	}
	G(1, 1) G(1, 2) G(1, 4) G(1, 8) G(1, 12)
	G(2, 1) G(2, 2) G(2, 4)
	G(4, 1) G(4, 2) G(4, 4)
#undef G
	return -1;
}

double power_sum(const std::vector<float> &a, const double *v, int n, int nrhs)
{
	double p = 0.0;
	for (int i = 0; i < n; i++)
		for (int c = 0; c < nrhs; c++) p += (double)a[i] * v[(size_t)i * nrhs + c];
	return p;
}

}  // namespace

// FP64 residual machinery: the caller's wT holds rp x ld doubles with rows
// >= nrhs and columns >= n zero; split-K partials; per-block stats.
struct Fx64 {
	int n = 0, ld = 0, nrhs = 0, rp = 0, rt = 1, ct = 1, W = 4, S = 1, ks = 1;
	Buf<double> part;
	size_t nblk = 0;
	double *blk = nullptr;  // the blocks' statistics, in host memory (Stage)

	int setup(int n_, int ld_, int nrhs_, Stage &stage, std::string &err)
	{
		n = n_;
		ld = ld_;
		nrhs = nrhs_;
		const int nct = (nrhs + 15) / 16;
		ct = nct >= 4 ? 4 : (nct >= 2 ? 2 : 1);
		rp = (nct + ct - 1) / ct * ct * 16;  // whole column groups: every tile the grid covers exists
		rt = 1;
		W = 4;
		S = 8;
		if (vec()) {
			// waves per row group (32 / ks rows a block): four below 8192 rows,
			// where fewer leave CUs without a block (n = 6144: 33.6, 31.8 and
			// 29.3 us at 1, 2 and 4; 4096: 22.5, 19.7, 16.6); above, as few as
			// fill the last round of 256 CUs to 95 % (less traffic of w per
			// row; us at 1, 2, 4: 8192 49.8, 59.1, 63.7; 9216 71.4, 67.6,
			// 61.9; 12288 102.4, 98.0, 98.5; 20224 259.7, 246.8, 262.5;
			// 32768 643, 667, 694)
			ks = 4;
			for (int k = 1; ld >= 8192 && k < 4; k *= 2) {
				const int blocks = ld / 32 * k, full = (blocks + 255) / 256 * 256;
				if (100 * blocks >= 95 * full) {
					ks = k;
					break;
				}
			}
			nblk = (size_t)ld / 32 * ks;
		} else {
			tile();
			launch_rows(n, nrhs, [&](auto, dim3 g) { nblk = g.x; });
			if (part.alloc((size_t)S * ld * rp, err)) return -1;
		}
		if (stage.stat_room(std::max<size_t>(nblk * 2, 3 * kStatBlocks), err)) return -1;
		blk = stage.stats;
		return 0;
	}
	// Row tiles per wave, waves per block and split-K of k_fx64m (ld is a
	// multiple of 256: every choice divides it).  Four column tiles: blocks of
	// 256 rows with the least split whose last round of 256 CUs is 85 % full, else
	// of 128 rows, else (small matrices) 64 rows split eight ways; fewer column
	// tiles: 128 rows from 4096 rows up for two, 64 rows for one, whose split
	// keeps the grid at 1024 blocks.  us at (rows per block, split), 64 columns, n
	// = 7936: (256, 8) 131, (128, 8) 149, (64, 8) 166; 192 columns, n = 4096: (256,
	// 8), a last round half full, 134, (128, 8) 103, (64, 8) 115; n = 1024: 21.5,
	// 14.1, 14.2; 32 columns, n = 2048: 12.0 at 128, 8.9 at 64.
	void tile()
	{
		const int groups = rp / (16 * ct);
		if (ct == 1) {
			while (S > 1 && ld / 64 * S > 1024) S /= 2;
		} else if (ct == 2) {
			W = ld >= 4096 ? 8 : 4;
		} else {
			for (int r = 2; r >= 1; r--)
				for (int s = 1; s <= 8; s *= 2) {
					const int blocks = ld / (128 * r) * groups * s, full = (blocks + 255) / 256 * 256;
					if (blocks >= 240 && 100 * blocks >= 85 * full) {
						rt = r;
						W = 8;
						S = s;
						return;
					}
				}
		}
	}
	// at most 4 columns: the vector-unit kernel
	bool vec() const { return nrhs <= 4; }
	template <int NC> void launch_vec(const float *F, const double *wT, const double *base, const double *rho,
	                                  const double *xT, double *out, hipStream_t st)
	{
		const dim3 g((unsigned)nblk), b(kB);
		if (ks == 1) hipLaunchKernelGGL((k_fx64v<NC, 1>), g, b, 0, st, F, wT, ld, n, xT, base, rho, out, blk);
		else if (ks == 2) hipLaunchKernelGGL((k_fx64v<NC, 2>), g, b, 0, st, F, wT, ld, n, xT, base, rho, out, blk);
		else hipLaunchKernelGGL((k_fx64v<NC, 4>), g, b, 0, st, F, wT, ld, n, xT, base, rho, out, blk);
	}
	// out = base + rho o (F w) - x (xT null: 0); returns (sum of squares, max |out|)
	int run(const float *F, const double *wT, const double *base, const double *rho, const double *xT, double *out,
	        hipStream_t st, double &ss, double &mx, bool want_stats, std::string &err)
	{
		if (vec()) {
			if (nrhs == 1) launch_vec<1>(F, wT, base, rho, xT, out, st);
			else if (nrhs == 2) launch_vec<2>(F, wT, base, rho, xT, out, st);
			else if (nrhs == 3) launch_vec<3>(F, wT, base, rho, xT, out, st);
			else launch_vec<4>(F, wT, base, rho, xT, out, st);
		} else {
			const dim3 grid(ld / (16 * rt * W), rp / (16 * ct), S), threads(64 * W);
			const int kchunk = ld / S;
			if (ct == 1) hipLaunchKernelGGL((k_fx64m<1, 1, 4>), grid, threads, 0, st, F, wT, part.p, ld, rp, kchunk);
			else if (ct == 2 && W == 4) hipLaunchKernelGGL((k_fx64m<1, 2, 4>), grid, threads, 0, st, F, wT, part.p, ld, rp, kchunk);
			else if (ct == 2) hipLaunchKernelGGL((k_fx64m<1, 2, 8>), grid, threads, 0, st, F, wT, part.p, ld, rp, kchunk);
			else if (W == 4) hipLaunchKernelGGL((k_fx64m<1, 4, 4>), grid, threads, 0, st, F, wT, part.p, ld, rp, kchunk);
			else if (rt == 1) hipLaunchKernelGGL((k_fx64m<1, 4, 8>), grid, threads, 0, st, F, wT, part.p, ld, rp, kchunk);
			else hipLaunchKernelGGL((k_fx64m<2, 4, 8>), grid, threads, 0, st, F, wT, part.p, ld, rp, kchunk);
			launch_rows(n, nrhs, [&](auto r, dim3 g) {
				hipLaunchKernelGGL(k_resid<decltype(r)::value>, g, dim3(kB), 0, st, part.p, S, ld, rp, n, nrhs, xT, base, rho,
				                   out, blk);
			});
		}
		HIP_OK(hipGetLastError(), "FP64 product");
		ss = mx = 0.0;
		if (!want_stats) return 0;
		HIP_OK(hipStreamSynchronize(st), "residual");
		for (size_t b = 0; b < nblk; b++) {
			ss += blk[2 * b];
			mx = std::max(mx, blk[2 * b + 1]);
		}
		return 0;
	}
};

// What a solve works in, kept between calls (grown where a wider one needs
// it).  Rows past the right-hand sides of xT, wT, X16 and Xb may hold an
// earlier call's columns, which touch only their own; columns past n are
// never written and stay zero.
struct Work {
	Buf<float> rho32, r32, part;
	Buf<double> rho64, E64, xT, wT, r64, out, fb, Bref64, blk;
	Buf<_Float16> X16[2];
	Buf<__bf16> Xb[2];
	Fx64 fx;
};

struct LinearSystem::Impl {
	hipStream_t st = nullptr;
	hipEvent_t e0 = nullptr, e1 = nullptr;
	Stage stage;
	Work work;
	Buf<float> F32, Ft, area;
	Buf<_Float16> F16, FT16;  // FT16: s16 * F^T in fragment order (the adjoint's sweeps)
	Buf<__bf16> FB16;
	Buf<unsigned> umax;
	const double *in[2] = {};  // inputs()
	float s16 = 1.f, sb16 = 1.f;
	bool have16 = false, haveb16 = false, havet = false, havet16 = false;
	std::map<std::pair<int, int>, std::pair<int, int>> tiles;  // (ct, prec) -> (rt, S)

	// low-precision fragment copy of F for prec (made once per matrix)
	int ensure_lowp(int prec, int ld, std::string &err)
	{
		const size_t npp = (size_t)ld * ld;
		if ((prec == PREC_F16 && have16) || (prec == PREC_BF16 && haveb16)) return 0;
		if (prec == PREC_F16) {
			if (umax.alloc(1, err)) return -1;
			HIP_OK(hipMemsetAsync(umax.p, 0, sizeof(unsigned), st), "memset");
			hipLaunchKernelGGL(k_absmax, dim3(4096), dim3(kB), 0, st, F32.p, npp, umax.p);
			unsigned bits = 0;
			HIP_OK(hipMemcpyAsync(&bits, umax.p, sizeof bits, hipMemcpyDeviceToHost, st), "absmax");
			HIP_OK(hipStreamSynchronize(st), "absmax");
			float m;
			std::memcpy(&m, &bits, sizeof m);
			if (!std::isfinite(m)) {
				err = "matrix has non-finite entries";
				return -1;
			}
			int e = 0;
			if (m > 0.f) e = std::max(-60, std::min(60, (int)std::floor(std::log2(16384.0 / m))));
			const float s = std::ldexp(1.0f, e);
			if (F16.alloc(npp, err)) return -1;
			hipLaunchKernelGGL(k_to_frag<_Float16>, dim3(8192), dim3(kB), 0, st, F32.p, ld, s, F16.p);
			s16 = s;
			have16 = true;
		} else if (prec == PREC_BF16) {
			if (FB16.alloc(npp, err)) return -1;
			hipLaunchKernelGGL(k_to_frag<__bf16>, dim3(8192), dim3(kB), 0, st, F32.p, ld, 1.0f, FB16.p);
			sb16 = 1.f;
			haveb16 = true;
		} else {
			err = "precision must be FP16 or BF16";
			return -1;
		}
		HIP_OK(hipGetLastError(), "convert");
		return 0;
	}
	// FP32 transpose of F (made once per matrix)
	int ensure_t(int ld, std::string &err)
	{
		if (havet) return 0;
		if (Ft.alloc((size_t)ld * ld, err)) return -1;
		hipLaunchKernelGGL(k_transpose, dim3(ld / 32, ld / 32), dim3(kB), 0, st, F32.p, Ft.p, ld);
		HIP_OK(hipGetLastError(), "transpose");
		havet = true;
		return 0;
	}
	// s16 * F^T in FP16 fragment order (made once per matrix)
	int ensure_t16(int ld, std::string &err)
	{
		if (havet16) return 0;
		if (ensure_lowp(PREC_F16, ld, err) || ensure_t(ld, err) || FT16.alloc((size_t)ld * ld, err)) return -1;
		hipLaunchKernelGGL(k_to_frag<_Float16>, dim3(8192), dim3(kB), 0, st, Ft.p, ld, s16, FT16.p);
		HIP_OK(hipGetLastError(), "convert");
		havet16 = true;
		return 0;
	}

	// the tile of a solve: tuned or forced, else by rule
	void solve_tile(int nrhs, int prec, int ld, int &rt, int &S) const
	{
		const auto t = tiles.find({pick_ct(nrhs), prec});
		if (t == tiles.end()) {
			sweep_tile(pick_ct(nrhs), ld, rt, S);
		} else {
			rt = t->second.first;
			S = t->second.second;
		}
	}

	// the start of a call: nothing of an earlier one (which may have ended in
	// an error) is in flight
	int begin(std::string &err)
	{
		HIP_OK(hipStreamSynchronize(st), "stream");
		stage.begin();
		return 0;
	}
	// rho and E (total each) where k_prep reads them: in pinned memory, or copied
	// to work.rho64 and E64
	int inputs(const double *rho, const double *E, size_t total, std::string &err)
	{
		double *h = (double *)stage.room(2 * total * 8);
		if (h) {
			std::memcpy(h, rho, total * 8);
			std::memcpy(h + total, E, total * 8);
			in[0] = h;
			in[1] = h + total;
			return 0;
		}
		in[0] = work.rho64.p;
		in[1] = work.E64.p;
		return stage.up(work.rho64.p, rho, total * 8, st, err) || stage.up(work.E64.p, E, total * 8, st, err) ? -1 : 0;
	}
	// room for count elements, zero where it was allocated anew
	template <typename T> int zeroed(Buf<T> &b, size_t count, std::string &err)
	{
		if (b.p && count <= b.n) return 0;
		if (b.alloc(count, err)) return -1;
		hipLaunchKernelGGL(k_fill<T>, dim3(grid_for(count)), dim3(kB), 0, st, b.p, count, (T)0.f);
		return 0;
	}
	// the iterate's two buffers (rp x ld, fragment order)
	template <typename E> int iterates(Buf<E> (&X)[2], size_t count, std::string &err)
	{
		return zeroed(X[0], count, err) || zeroed(X[1], count, err) ? -1 : 0;
	}
	template <typename E> Buf<E> (&iterate_of())[2]
	{
		if constexpr (std::is_same_v<E, _Float16>) return work.X16;
		else return work.Xb;
	}
	double power(size_t blocks) const
	{
		double p = 0.0;
		for (size_t b = 0; b < blocks; b++) p += stage.stats[b];
		return p;
	}

	// times one sweep for every (rows per wave, split-K) and keeps the fastest
	template <typename E> int tune(const E *A, int n, int ld, int nrhs, int prec, std::string &err)
	{
		const int ct = pick_ct(nrhs), rp = ct * 16;
		const size_t total = (size_t)n * nrhs;
		Buf<E> X[2];
		Buf<float> part, r32, rho;
		if (iterates(X, (size_t)rp * ld, err) || r32.alloc(total, err) || rho.alloc(total, err) ||
		    (ct >= 8 && part.alloc((size_t)8 * ld * rp, err)))
			return -1;
		hipLaunchKernelGGL(k_fill<float>, dim3(grid_for(total)), dim3(kB), 0, st, r32.p, total, 1.0f);
		hipLaunchKernelGGL(k_fill<float>, dim3(grid_for(total)), dim3(kB), 0, st, rho.p, total, 0.5f);
		SweepOut<E> o{};
		o.n = n, o.nrhs = nrhs, o.inv = 1.0f, o.rhs = r32.p, o.rho = rho.p, o.XTn = X[1].p;
		double best = 1e30;
		int brt = 0, bs = 0;
		for (int rt : {1, 2, 4}) {
			for (int S : {1, 2, 4, 8}) {
				if (launch_sweep<E>(rt, ct, S, A, X[0].p, part.p, ld, rp, o, st)) continue;  // warm-up
				HIP_OK(hipEventRecord(e0, st), "event");
				for (int k = 0; k < 3; k++) launch_sweep<E>(rt, ct, S, A, X[0].p, part.p, ld, rp, o, st);
				HIP_OK(hipEventRecord(e1, st), "event");
				HIP_OK(hipEventSynchronize(e1), "event");
				float ms = 0;
				HIP_OK(hipEventElapsedTime(&ms, e0, e1), "event");
				if (ms < best) {
					best = ms;
					brt = rt;
					bs = S;
				}
			}
		}
		HIP_OK(hipGetLastError(), "autotune");
		HIP_OK(hipStreamSynchronize(st), "autotune");
		if (!brt) {
			err = "autotune: no valid tile";
			return -1;
		}
		tiles[{ct, prec}] = {brt, bs};
		return 0;
	}

	template <typename E>
	int time_product(const E *A, int n, int ld, int nrhs, int prec, int reps, double *ms, std::string &err)
	{
		const int ct = pick_ct(nrhs), rp = ct * 16;
		const auto [rt, S] = tiles.at({ct, prec});
		const size_t total = (size_t)n * nrhs, xts = (size_t)rp * ld;
		Buf<E> x;
		Buf<float> part, y;
		if (x.alloc(xts, err) || y.alloc(total, err) || (dma_tile(rt, ct) && part.alloc((size_t)S * ld * rp, err)))
			return -1;
		hipLaunchKernelGGL(k_fill<E>, dim3(grid_for(xts)), dim3(kB), 0, st, x.p, xts, (E)1.f);
		SweepOut<E> o{};
		o.n = n, o.nrhs = nrhs, o.inv = 1.0f, o.y = y.p;
		launch_sweep<E>(rt, ct, S, A, x.p, part.p, ld, rp, o, st, false);
		HIP_OK(hipEventRecord(e0, st), "event");
		for (int k = 0; k < reps; k++) launch_sweep<E>(rt, ct, S, A, x.p, part.p, ld, rp, o, st, false);
		HIP_OK(hipEventRecord(e1, st), "event");
		HIP_OK(hipEventSynchronize(e1), "event");
		HIP_OK(hipGetLastError(), "gemm_ms");
		float t = 0;
		HIP_OK(hipEventElapsedTime(&t, e0, e1), "event");
		*ms = t / reps;
		return 0;
	}

	// Y = F X in prec; the tuned or forced tile, else one wave per 16 rows
	template <typename E>
	int product(const E *A, float inv, int n, int ld, int nrhs, int prec, const double *X, double *Y, std::string &err)
	{
		const int ct = pick_ct(nrhs), rp = ct * 16;
		int rt = 1, S = 1;
		if (const auto it = tiles.find({ct, prec}); it != tiles.end()) {
			rt = it->second.first;
			S = it->second.second;
		}
		const size_t total = (size_t)n * nrhs, xts = (size_t)rp * ld;
		Work &w = work;
		Buf<E>(&x)[2] = iterate_of<E>();
		if (begin(err) || iterates(x, xts, err) || w.r32.alloc(total, err) || w.E64.alloc(total, err) ||
		    (dma_tile(rt, ct) && w.part.alloc((size_t)S * ld * rp, err)) || stage.up(w.E64.p, X, total * 8, st, err))
			return -1;
		launch_scale(w.E64.p, 1.0, n, nrhs, ld, w.r32.p, x[0].p, nullptr, st);
		SweepOut<E> o{};
		o.n = n, o.nrhs = nrhs, o.inv = inv, o.y = w.r32.p;
		if (launch_sweep<E>(rt, ct, S, A, x[0].p, w.part.p, ld, rp, o, st)) {
			err = "multiply: no kernel for this tile";
			return -1;
		}
		HIP_OK(hipGetLastError(), "multiply");
		std::vector<float> hy(total);
		if (stage.down(hy.data(), w.r32.p, total * 4, st, err)) return -1;
		for (size_t t = 0; t < total; t++) Y[t] = hy[t];
		return 0;
	}

	// the sweeps of one refinement (v <- rhs + .. from X[0]); the last one
	// adds the correction to the iterate
	template <typename E>
	int sweep(const E *A, Buf<E> (&X)[2], float *part, int ct, int rt, int S, int ld, int sweeps, SweepOut<E> o,
	          std::string &err)
	{
		double *xT = o.xT;
		for (int m = 0; m < sweeps; m++) {
			o.XTn = X[(m + 1) & 1].p;
			o.xT = m == sweeps - 1 ? xT : nullptr;
			if (launch_sweep<E>(rt, ct, S, A, X[m & 1].p, part, ld, ct * 16, o, st)) {
				err = "no kernel for this tile";
				return -1;
			}
		}
		return 0;
	}
};

LinearSystem::~LinearSystem()
{
	if (!d_) return;
	if (d_->st) (void)hipStreamSynchronize(d_->st);
	if (d_->e0) (void)hipEventDestroy(d_->e0);
	if (d_->e1) (void)hipEventDestroy(d_->e1);
	hipStream_t s = d_->st;
	delete d_;
	if (s) (void)hipStreamDestroy(s);
}

LinearSystem *LinearSystem::create(int n, std::string &err)
{
	if (n <= 0 || n > (1 << 17)) {
		err = "linear system size must be 1..131072";
		return nullptr;
	}
	int ndev = 0;
	if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
		err = "no HIP device available";
		return nullptr;
	}
	LinearSystem *L = new LinearSystem();
	L->d_ = new Impl();
	L->n_ = n;
	L->np_ = (n + 255) / 256 * 256;
	const size_t np = L->np_;
	if (hipStreamCreateWithFlags(&L->d_->st, hipStreamNonBlocking) != hipSuccess ||
	    hipEventCreate(&L->d_->e0) != hipSuccess || hipEventCreate(&L->d_->e1) != hipSuccess) {
		err = "stream/event creation failed";
		delete L;
		return nullptr;
	}
	if (L->d_->F32.alloc(np * np, err) || hipMemset(L->d_->F32.p, 0, np * np * sizeof(float)) != hipSuccess) {
		if (err.empty()) err = "matrix clear failed";
		delete L;
		return nullptr;
	}
	if (L->d_->stage.init(err)) {
		delete L;
		return nullptr;
	}
	std::vector<float> ones(n, 1.0f);
	if (L->d_->area.alloc(n, err) ||
	    hipMemcpy(L->d_->area.p, ones.data(), n * sizeof(float), hipMemcpyHostToDevice) != hipSuccess) {
		if (err.empty()) err = "area upload failed";
		delete L;
		return nullptr;
	}
	return L;
}

float *LinearSystem::matrix32()
{
	d_->have16 = d_->haveb16 = d_->havet = d_->havet16 = false;  // the caller may rewrite F
	return d_->F32.p;
}

void *LinearSystem::stream() const { return (void *)d_->st; }

int LinearSystem::set_matrix(const float *F, std::string &err)
{
	HIP_OK(hipMemcpy2D(matrix32(), (size_t)np_ * 4, F, (size_t)n_ * 4, (size_t)n_ * 4, n_, hipMemcpyHostToDevice),
	       "set matrix");
	return 0;
}

int LinearSystem::get_matrix(float *F, std::string &err)
{
	HIP_OK(hipMemcpy2D(F, (size_t)n_ * 4, d_->F32.p, (size_t)np_ * 4, (size_t)n_ * 4, n_, hipMemcpyDeviceToHost),
	       "get matrix");
	return 0;
}

int LinearSystem::set_areas(const double *area, std::string &err)
{
	std::vector<float> a(n_);
	for (int i = 0; i < n_; i++) a[i] = (float)area[i];
	HIP_OK(hipMemcpy(d_->area.p, a.data(), n_ * sizeof(float), hipMemcpyHostToDevice), "set areas");
	return 0;
}

void LinearSystem::tile_config(int nrhs, int prec, int *rt, int *splitk) const
{
	const int ct = pick_ct(nrhs);
	auto it = d_->tiles.find({ct, prec});
	if (it == d_->tiles.end()) {
		*rt = 0;
		*splitk = 0;
	} else {
		*rt = it->second.first;
		*splitk = it->second.second;
	}
}

int LinearSystem::set_tile(int nrhs, int prec, int rt, int splitk, std::string &err)
{
	const int ct = pick_ct(nrhs);
	if (nrhs <= 0 || ct < 0 || (prec != PREC_F16 && prec != PREC_BF16) || (rt != 1 && rt != 2 && rt != 4) ||
	    (splitk != 1 && splitk != 2 && splitk != 4 && splitk != 8)) {
		err = "set_tile: nrhs 1..192, precision FP16 or BF16, rt 1, 2 or 4, splitk 1, 2, 4 or 8";
		return -1;
	}
	d_->tiles[{ct, prec}] = {rt, splitk};
	return 0;
}

// Times one sweep for every (rows per wave, split-K) and keeps the fastest for
// (nrhs column tiles, precision).
int LinearSystem::autotune(int nrhs, int prec, std::string &err)
{
	Impl &d = *d_;
	const int ct = pick_ct(nrhs);
	if (nrhs <= 0 || ct < 0 || (prec != PREC_F16 && prec != PREC_BF16)) {
		err = "autotune: nrhs must be 1..192 and precision FP16 or BF16";
		return -1;
	}
	if (d.ensure_lowp(prec, np_, err)) return -1;
	const int rc = prec == PREC_F16 ? d.tune<_Float16>(d.F16.p, n_, np_, nrhs, prec, err)
	                                : d.tune<__bf16>(d.FB16.p, n_, np_, nrhs, prec, err);
	return rc;
}


int LinearSystem::gemm_ms(int nrhs, int prec, int reps, double *ms, std::string &err)
{
	Impl &d = *d_;
	const int ct = pick_ct(nrhs);
	if (nrhs <= 0 || ct < 0 || (prec != PREC_F16 && prec != PREC_BF16) || reps <= 0) {
		err = "gemm_ms: bad arguments";
		return -1;
	}
	if (!d.tiles.count({ct, prec}) && autotune(nrhs, prec, err)) return -1;
	if (d.ensure_lowp(prec, np_, err)) return -1;
	return prec == PREC_F16 ? d.time_product<_Float16>(d.F16.p, n_, np_, nrhs, prec, reps, ms, err)
	                        : d.time_product<__bf16>(d.FB16.p, n_, np_, nrhs, prec, reps, ms, err);
}

int LinearSystem::multiply(int prec, int nrhs, const double *X, double *Y, std::string &err)
{
	Impl &d = *d_;
	const int ct = pick_ct(nrhs);
	if (nrhs <= 0 || ct < 0) {
		err = "multiply: nrhs must be 1..192";
		return -1;
	}
	const int n = n_, ld = np_;
	const size_t total = (size_t)n * nrhs;
	hipStream_t st = d.st;
	if (prec == PREC_F32) {
		Work &w = d.work;
		if (d.begin(err) || w.fx.setup(n, ld, nrhs, d.stage, err) || d.zeroed(w.xT, (size_t)w.fx.rp * ld, err) ||
		    w.E64.alloc(total, err) || w.out.alloc(total, err) || d.stage.up(w.E64.p, X, total * 8, st, err))
			return -1;
		hipLaunchKernelGGL(k_cols, turn_grid(n, nrhs), dim3(kB), 0, st, w.E64.p, ld, n, nrhs, w.xT.p);
		double ss, mx;
		if (w.fx.run(d.F32.p, w.xT.p, nullptr, nullptr, nullptr, w.out.p, st, ss, mx, false, err)) return -1;
		return d.stage.down(Y, w.out.p, total * 8, st, err);
	}
	if (d.ensure_lowp(prec, ld, err)) return -1;
	return prec == PREC_F16 ? d.product<_Float16>(d.F16.p, 1.0f / d.s16, n, ld, nrhs, prec, X, Y, err)
	                        : d.product<__bf16>(d.FB16.p, 1.0f / d.sb16, n, ld, nrhs, prec, X, Y, err);
}

int LinearSystem::gather(int prec, int nrhs, const double *rho, const double *E, double tol, int max_outer, int sweeps,
                         const double *Bref, double target, double *B, double *info, std::string &err)
{
	Impl &d = *d_;
	const int ct = pick_ct(nrhs);
	if (nrhs <= 0 || ct < 0) {
		err = "gather: nrhs must be 1..192";
		return -1;
	}
	if (prec != PREC_F16 && prec != PREC_BF16) {
		err = "gather: precision must be FP16 or BF16";
		return -1;
	}
	if (sweeps <= 0 || max_outer < 0) {
		err = "gather: sweeps must be > 0 and max_outer >= 0";
		return -1;
	}
	if (d.ensure_lowp(prec, np_, err)) return -1;
	int rt, S;
	d.solve_tile(nrhs, prec, np_, rt, S);
	const int n = n_, ld = np_, rp = ct * 16;
	const size_t total = (size_t)n * nrhs;
	const float inv = 1.0f / (prec == PREC_F16 ? d.s16 : d.sb16);
	hipStream_t st = d.st;
	Work &w = d.work;
	const size_t xts = (size_t)rp * ld;
	if (d.begin(err) || w.fx.setup(n, ld, nrhs, d.stage, err) || w.rho32.alloc(total, err) || w.r32.alloc(total, err) ||
	    (dma_tile(rt, ct) && w.part.alloc((size_t)S * ld * rp, err)) || w.rho64.alloc(total, err) ||
	    w.E64.alloc(total, err) || d.zeroed(w.xT, (size_t)w.fx.rp * ld, err) || w.r64.alloc(total, err) ||
	    w.out.alloc(total, err) || (prec == PREC_F16 ? d.iterates(w.X16, xts, err) : d.iterates(w.Xb, xts, err)) ||
	    d.inputs(rho, E, total, err))
		return -1;
	if (Bref && (w.Bref64.alloc(total, err) || w.blk.alloc(8192 * 2, err) ||
	             d.stage.up(w.Bref64.p, Bref, total * 8, st, err)))
		return -1;
	const int g = grid_for(total), gs = std::min(g, kStatBlocks);
	hipLaunchKernelGGL(k_prep, dim3(gs), dim3(kB), 0, st, d.in[0], d.in[1], d.area.p, (unsigned)total, (unsigned)nrhs,
	                   w.rho32.p, d.stage.stats, w.rho64.p, w.E64.p);
	HIP_OK(hipGetLastError(), "upload");
	HIP_OK(hipStreamSynchronize(st), "upload");
	d.stage.begin();  // the inputs were read
	// x = 0 at the start, so the first residual is E itself
	double ss0 = 0.0, mx0 = 0.0, power_E = 0.0;
	for (int k = 0; k < gs; k++) {
		ss0 += d.stage.stats[3 * k];
		mx0 = std::max(mx0, d.stage.stats[3 * k + 1]);
		power_E += d.stage.stats[3 * k + 2];
	}
	std::vector<double> hb(Bref ? 8192 * 2 : 0);
	auto err_vs_ref = [&](double &e) -> int {
		hipLaunchKernelGGL(k_err, dim3(g), dim3(kB), 0, st, w.xT.p, 1, ld, w.Bref64.p, n, nrhs, w.blk.p);
		HIP_OK(hipMemcpyAsync(hb.data(), w.blk.p, (size_t)g * 2 * 8, hipMemcpyDeviceToHost, st), "err");
		HIP_OK(hipStreamSynchronize(st), "err");
		double a = 0.0, b = 0.0;
		for (int k = 0; k < g; k++) {
			a += hb[2 * k];
			b += hb[2 * k + 1];
		}
		e = std::sqrt(a / std::max(b, 1e-300));
		return 0;
	};
	const auto t0 = std::chrono::steady_clock::now();
	double enorm = -1.0, rel = 0.0, ms_target = -1.0, errv = -1.0, check_ms = 0.0;
	int outer = 0, total_sweeps = 0;
	for (;; outer++) {
		double ss = ss0, mx = mx0;
		if (outer > 0 && w.fx.run(d.F32.p, w.xT.p, w.E64.p, w.rho64.p, w.xT.p, w.r64.p, st, ss, mx, true, err)) return -1;
		if (!std::isfinite(ss)) {
			err = "gather diverged (non-finite residual): the iteration needs spectral radius of diag(rho) F below 1";
			return -1;
		}
		if (enorm < 0) enorm = std::sqrt(ss);  // x = 0: the first residual is E
		rel = enorm > 0 ? std::sqrt(ss) / enorm : 0.0;
		if (Bref && outer > 0) {
			const auto c0 = std::chrono::steady_clock::now();
			if (err_vs_ref(errv)) return -1;
			check_ms += ms_since(c0);
			if (ms_target < 0 && errv <= target) ms_target = ms_since(t0) - check_ms;
		}
		if (rel <= tol || outer >= max_outer || mx == 0.0) break;
		const double s = mx;
		int rc;
		auto refine = [&](const auto *A, auto &X) {
			typedef std::remove_cv_t<std::remove_pointer_t<decltype(A)>> T;
			launch_scale(outer ? w.r64.p : w.E64.p, 1.0 / s, n, nrhs, ld, w.r32.p, X[0].p, nullptr, st);
			SweepOut<T> o{};
			o.n = n, o.nrhs = nrhs, o.inv = inv, o.rhs = w.r32.p, o.rho = w.rho32.p;
			o.xT = w.xT.p, o.s = s, o.first = outer == 0;
			rc = d.sweep(A, X, w.part.p, ct, rt, S, ld, sweeps, o, err);
		};
		if (prec == PREC_F16) refine(d.F16.p, w.X16);
		else refine(d.FB16.p, w.Xb);
		if (rc) return -1;
		total_sweeps += sweeps;
		HIP_OK(hipGetLastError(), "sweep launch");
	}
	const double ms = ms_since(t0) - check_ms;
	if (outer == 0)  // no refinement: the iterate is the zero it started from
		hipLaunchKernelGGL(k_fill<double>, dim3(grid_for(w.xT.n)), dim3(kB), 0, st, w.xT.p, w.xT.n, 0.0);
	const dim3 tg = turn_grid(n, nrhs);
	const size_t blocks = (size_t)tg.x * tg.y;
	if (d.stage.stat_room(blocks, err)) return -1;  // the residual's were read
	double *out = (double *)d.stage.room(total * 8);
	hipLaunchKernelGGL(k_rows, tg, dim3(kB), 0, st, w.xT.p, ld, n, nrhs, nullptr, out ? out : w.out.p, d.area.p,
	                   d.stage.stats);
	HIP_OK(hipGetLastError(), "download");
	if (out) {
		HIP_OK(hipStreamSynchronize(st), "download");
		std::memcpy(B, out, total * 8);
	} else if (d.stage.down(B, w.out.p, total * 8, st, err)) {
		return -1;
	}
	if (info) {
		info[INFO_OUTER] = outer;
		info[INFO_SWEEPS] = total_sweeps;
		info[INFO_REL_RES] = rel;
		info[INFO_MS] = ms;
		info[INFO_MS_TARGET] = ms_target;
		info[INFO_ERR] = errv;
		info[INFO_POWER_E] = power_E;
		info[INFO_POWER_B] = d.power(blocks);
	}
	return 0;
}

int LinearSystem::shoot(int nrhs, const double *rho, const double *E, const double *Bref, double target, int max_shots,
                        double *B, double *info, std::string &err)
{
	Impl &d = *d_;
	if (nrhs <= 0 || nrhs > kMaxShootRhs) {
		err = "shoot: nrhs must be 1..16";
		return -1;
	}
	if (max_shots < 0) {
		err = "shoot: max_shots must be >= 0";
		return -1;
	}
	const int n = n_, ld = np_;
	hipStream_t st = d.st;
	static_assert(sizeof(ShotRec) % 8 == 0, "record alignment");
	if (d.ensure_t(ld, err)) return -1;
	const size_t total = (size_t)n * nrhs;
	const int nb = (n + kB - 1) / kB;
	Buf<float> rho32, B32, dB32;
	Buf<ShotRec> rec;
	Buf<int> shots_d;
	if (rho32.alloc(total, err) || B32.alloc(total, err) || dB32.alloc(total, err) || rec.alloc(2 * (size_t)nb, err) ||
	    shots_d.alloc(1, err))
		return -1;
	std::vector<float> h(total);
	for (size_t t = 0; t < total; t++) h[t] = (float)rho[t];
	HIP_OK(hipMemcpyAsync(rho32.p, h.data(), total * 4, hipMemcpyHostToDevice, st), "upload");
	std::vector<float> e32(total);
	for (size_t t = 0; t < total; t++) e32[t] = (float)E[t];
	HIP_OK(hipMemcpyAsync(B32.p, e32.data(), total * 4, hipMemcpyHostToDevice, st), "upload");
	HIP_OK(hipMemcpyAsync(dB32.p, e32.data(), total * 4, hipMemcpyHostToDevice, st), "upload");
	hipLaunchKernelGGL(k_fill<int>, dim3(1), dim3(kB), 0, st, shots_d.p, (size_t)1, 0);
	HIP_OK(hipStreamSynchronize(st), "upload");
	std::vector<float> hb(total);
	auto err_vs_ref = [&](double &e) -> int {
		HIP_OK(hipMemcpyAsync(hb.data(), B32.p, total * 4, hipMemcpyDeviceToHost, st), "err");
		HIP_OK(hipStreamSynchronize(st), "err");
		double a = 0.0, b = 0.0;
		for (size_t t = 0; t < total; t++) {
			const double x = (double)hb[t] - Bref[t];
			a += x * x;
			b += Bref[t] * Bref[t];
		}
		e = std::sqrt(a / std::max(b, 1e-300));
		return 0;
	};
	// shot k reads the records of shot k - 1 (parity k & 1) and writes the
	// other set
	auto launch_shot = [&](int k) {
		hipLaunchKernelGGL(k_lshoot, dim3(nb), dim3(kB), 0, st, d.Ft.p, ld, rho32.p, d.area.p, B32.p, dB32.p, n, nrhs,
		                   rec.p + (size_t)(k & 1) * nb, rec.p + (size_t)((k + 1) & 1) * nb, shots_d.p);
	};
	// Where one block holds the system, a launch makes many shots; else a shot
	// needs the previous launch's argmax and plain shooting is bound by launch
	// latency: runs of kGraphShots shots (an even number, so parities repeat)
	// are captured once into a HIP graph and replayed.
	constexpr int kGraphShots = 64;
	struct GraphGuard {
		hipGraph_t g = nullptr;
		hipGraphExec_t x = nullptr;
		~GraphGuard()
		{
			if (x) (void)hipGraphExecDestroy(x);
			if (g) (void)hipGraphDestroy(g);
		}
	} run;
	auto one = [&](int shots) {
		return launch_shoot_one(d.Ft.p, ld, rho32.p, d.area.p, B32.p, dB32.p, n, nrhs, shots, shots_d.p, st);
	};
	const bool single = one(0);  // no shot: whether there is a kernel for the size
	if (!single) {
		HIP_OK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), "shot capture");
		for (int k = 0; k < kGraphShots; k++) launch_shot(k);
		HIP_OK(hipStreamEndCapture(st, &run.g), "shot capture");
		HIP_OK(hipGraphInstantiate(&run.x, run.g, nullptr, nullptr, 0), "shot graph");
	}
	const auto t0 = std::chrono::steady_clock::now();
	if (!single)
		hipLaunchKernelGGL(k_lsel, dim3(nb), dim3(kB), 0, st, dB32.p, d.area.p, n, nrhs, rec.p);
	double check_ms = 0.0, ms_target = -1.0, errv = -1.0;
	// shots per look at the state: as many as the error against Bref may be
	// late by; with none to check, a launch of the one-block kernel ends by itself
	int launched = 0, chunk = single && !Bref ? 4096 : 64, done_shots = 0;
	for (;;) {
		const int b = std::min(chunk, max_shots - launched);
		if (b <= 0) break;
		if (single) {
			one(b);
		} else {
			int k = 0;
			if ((launched & 1) == 0)
				for (; k + kGraphShots <= b; k += kGraphShots) HIP_OK(hipGraphLaunch(run.x, st), "shot graph launch");
			for (; k < b; k++) launch_shot(launched + k);
		}
		launched += b;
		HIP_OK(hipGetLastError(), "shoot launch");
		HIP_OK(hipMemcpyAsync(&done_shots, shots_d.p, sizeof(int), hipMemcpyDeviceToHost, st), "state");
		HIP_OK(hipStreamSynchronize(st), "shoot");
		if (Bref) {
			const auto c0 = std::chrono::steady_clock::now();
			if (err_vs_ref(errv)) return -1;
			check_ms += ms_since(c0);
			if (errv <= target) {
				ms_target = ms_since(t0) - check_ms;
				break;
			}
		}
		if (done_shots < launched) break;  // a launch found nothing left to shoot
		chunk = std::min(chunk * 2, 4096);
	}
	const double ms = ms_since(t0) - check_ms;
	HIP_OK(hipMemcpy(hb.data(), B32.p, total * 4, hipMemcpyDeviceToHost), "download");
	for (size_t t = 0; t < total; t++) B[t] = hb[t];
	if (Bref && errv < 0 && err_vs_ref(errv)) return -1;
	if (info) {
		std::vector<float> a(n);
		HIP_OK(hipMemcpy(a.data(), d.area.p, n * 4, hipMemcpyDeviceToHost), "area");
		info[INFO_OUTER] = done_shots;
		info[INFO_SWEEPS] = 0;
		info[INFO_REL_RES] = -1;
		info[INFO_MS] = ms;
		info[INFO_MS_TARGET] = ms_target;
		info[INFO_ERR] = errv;
		info[INFO_POWER_E] = power_sum(a, E, n, nrhs);
		info[INFO_POWER_B] = power_sum(a, B, n, nrhs);
	}
	return 0;
}

int LinearSystem::adjoint(int nrhs, const double *rho, const double *B, const double *gin, double tol, int max_outer,
                          int sweeps, double *lambda, double *drho, double *info, std::string &err)
{
	Impl &d = *d_;
	if (nrhs <= 0 || nrhs > 4) {
		err = "adjoint: nrhs must be 1..4";
		return -1;
	}
	if (sweeps <= 0 || max_outer < 0) {
		err = "adjoint: sweeps must be > 0 and max_outer >= 0";
		return -1;
	}
	const int n = n_, ld = np_;
	const size_t total = (size_t)n * nrhs;
	hipStream_t st = d.st;
	// the sweeps multiply by F^T in FP16 on MFMA (the gather's kernels on
	// the transposed fragment copy); the residual stays FP64 over FP32 F
	const int ct = pick_ct(nrhs), rp = ct * 16;
	if (d.ensure_t16(ld, err)) return -1;
	int rt, Sg;
	d.solve_tile(nrhs, PREC_F16, ld, rt, Sg);
	const float inv = 1.0f / d.s16;
	const int g = grid_for(total), gs = std::min(g, kStatBlocks);
	Work &w = d.work;
	if (d.begin(err) || w.fx.setup(n, ld, nrhs, d.stage, err)) return -1;
	const size_t xtn = (size_t)w.fx.rp * ld;
	// out: lambda, then dL/drho
	if (w.rho64.alloc(total, err) || w.E64.alloc(total, err) || d.zeroed(w.xT, xtn, err) || d.zeroed(w.wT, xtn, err) ||
	    w.r64.alloc(total, err) || w.out.alloc(2 * total, err) || w.rho32.alloc(total, err) || w.r32.alloc(total, err) ||
	    w.fb.alloc(total, err) || d.iterates(w.X16, (size_t)rp * ld, err) || d.inputs(rho, gin, total, err))
		return -1;
	hipLaunchKernelGGL(k_prep, dim3(gs), dim3(kB), 0, st, d.in[0], d.in[1], d.area.p, (unsigned)total, (unsigned)nrhs,
	                   w.rho32.p, d.stage.stats, w.rho64.p, w.E64.p);
	HIP_OK(hipGetLastError(), "upload");
	HIP_OK(hipStreamSynchronize(st), "upload");
	d.stage.begin();  // the inputs were read
	const auto t0 = std::chrono::steady_clock::now();
	double enorm = -1.0, rel = 0.0;
	int outer = 0, total_sweeps = 0;
	double ss0 = 0.0, mx0 = 0.0;  // lambda = 0 at the start: the first residual is g
	for (int k = 0; k < gs; k++) {
		ss0 += d.stage.stats[3 * k];
		mx0 = std::max(mx0, d.stage.stats[3 * k + 1]);
	}
	for (;; outer++) {
		double ss = ss0, mx = mx0;
		// r = g + F^T (rho o x) - x in FP64 over the transposed copy that the
		// FP16 one is made from: its rows are read whole, where F's columns,
		// split over row chunks, ran at a sixth of the rate (n = 6001: 151 +
		// 8.6 -> 29 us)
		if (outer > 0 && w.fx.run(d.Ft.p, w.wT.p, w.E64.p, nullptr, w.xT.p, w.r64.p, st, ss, mx, true, err)) return -1;
		if (!std::isfinite(ss)) {
			err = "adjoint diverged (non-finite residual)";
			return -1;
		}
		if (enorm < 0) enorm = std::sqrt(ss);
		rel = enorm > 0 ? std::sqrt(ss) / enorm : 0.0;
		if (rel <= tol || outer >= max_outer || mx == 0.0) break;
		// d <- r (scaled), then sweeps d <- r + F^T (rho o d) with XT = rho o d
		launch_scale(outer ? w.r64.p : w.E64.p, 1.0 / mx, n, nrhs, ld, w.r32.p, w.X16[0].p, w.rho32.p, st);
		SweepOut<_Float16> o{};
		o.n = n, o.nrhs = nrhs, o.inv = inv, o.rho_in = true, o.rhs = w.r32.p, o.rho = w.rho32.p;
		o.xT = w.xT.p, o.s = mx, o.first = outer == 0, o.wT = w.wT.p, o.rho64 = w.rho64.p;
		if (d.sweep(d.FT16.p, w.X16, nullptr, ct, rt, Sg, ld, sweeps, o, err)) return -1;
		total_sweeps += sweeps;
		HIP_OK(hipGetLastError(), "adjoint sweep");
	}
	if (outer == 0)  // no refinement: lambda is the zero it started from
		hipLaunchKernelGGL(k_fill<double>, dim3(grid_for(w.xT.n)), dim3(kB), 0, st, w.xT.p, w.xT.n, 0.0);
	// dL/drho = lambda o (F B), F B in FP64 (wT takes B)
	double *hB = (double *)d.stage.room(total * 8);
	if (hB) std::memcpy(hB, B, total * 8);
	else if (d.stage.up(w.r64.p, B, total * 8, st, err)) return -1;
	const dim3 tg = turn_grid(n, nrhs);
	hipLaunchKernelGGL(k_cols, tg, dim3(kB), 0, st, hB ? hB : w.r64.p, ld, n, nrhs, w.wT.p);
	{
		double ss, mx;
		if (w.fx.run(d.F32.p, w.wT.p, nullptr, nullptr, nullptr, w.fb.p, st, ss, mx, false, err)) return -1;
	}
	double *out = (double *)d.stage.room(2 * total * 8), *o = out ? out : w.out.p;
	hipLaunchKernelGGL(k_rows, tg, dim3(kB), 0, st, w.xT.p, ld, n, nrhs, nullptr, o, nullptr, nullptr);
	hipLaunchKernelGGL(k_rows, tg, dim3(kB), 0, st, w.xT.p, ld, n, nrhs, w.fb.p, o + total, nullptr, nullptr);
	HIP_OK(hipGetLastError(), "adjoint");
	if (out) {
		HIP_OK(hipStreamSynchronize(st), "adjoint");
		std::memcpy(lambda, out, total * 8);
		std::memcpy(drho, out + total, total * 8);
	} else {
		const Stage::Part parts[2] = {{lambda, total * 8}, {drho, total * 8}};
		if (d.stage.down_parts(w.out.p, parts, 2, st, err)) return -1;
	}
	const double ms = ms_since(t0);
	if (info) {
		for (int k = 0; k < INFO_N; k++) info[k] = -1;
		info[INFO_OUTER] = outer;
		info[INFO_SWEEPS] = total_sweeps;
		info[INFO_REL_RES] = rel;
		info[INFO_MS] = ms;
	}
	return 0;
}

}  // namespace rgpu
