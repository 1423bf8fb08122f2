// Device building blocks shared by the explicit-matrix solvers (linear.hip)
// and the batched solver (batch.hip): MFMA fragment layout, the
// sweep, the FP64 residual of few columns, buffers.
// Included inside an anonymous namespace of each translation unit.
#pragma once

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kB = 256;

__device__ __forceinline__ f4 mfma(h8 a, h8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ f4 mfma(b8 a, b8 b, f4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }

template <typename E> struct VecOf;
template <> struct VecOf<_Float16> { typedef h8 type; };
template <> struct VecOf<__bf16> { typedef b8 type; };

// element (row, k) of a fragment-ordered matrix with ld columns
__device__ __forceinline__ size_t frag_index(int row, int k, int ld)
{
	return ((size_t)(row >> 4) * (ld >> 5) + (k >> 5)) * 512 + ((((k & 31) >> 3) << 4) + (row & 15)) * 8 + (k & 7);
}

// entries (c, i .. i + R - 1), R 1 or 8 and i a multiple of it
template <int R, typename E> __device__ __forceinline__ void put_frag(E *XT, int c, int i, int ld, const E (&x)[R])
{
	typedef typename VecOf<E>::type V;
	static_assert(R == 1 || R == 8, "an entry or a fragment row");
	E *o = XT + frag_index(c, i, ld);
	if constexpr (R == 1) {
		*o = x[0];
	} else {
		V v;
#pragma unroll
		for (int r = 0; r < R; r++) v[r] = x[r];
		*(V *)o = v;
	}
}

// the largest |F|, of count (a multiple of 4) entries: NaN is passed over.  One
// atomic per wave was 189 us at any size: n = 1000 189 -> 14, 9000 237 -> 71,
// 20000 530 -> 315 us (5.1 TB/s).
__global__ __launch_bounds__(kB) void k_absmax(const float *F, size_t count, unsigned *out)
{
	const float4 *v = (const float4 *)F;
	const size_t n4 = count / 4, step = (size_t)gridDim.x * kB;
	float m = 0.f;
	auto take = [&](const float4 &a) { m = fmaxf(m, fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w)))); };
	size_t i = blockIdx.x * (size_t)kB + threadIdx.x;
	for (; i + 3 * step < n4; i += 4 * step) {  // four loads in flight
		const float4 a = v[i], b = v[i + step], c = v[i + 2 * step], d = v[i + 3 * step];
		take(a);
		take(b);
		take(c);
		take(d);
	}
	for (; i < n4; i += step) take(v[i]);
	for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
	__shared__ float w[kB / 64];
	if ((threadIdx.x & 63) == 0) w[threadIdx.x >> 6] = m;
	__syncthreads();
	m = fmaxf(fmaxf(w[0], w[1]), fmaxf(w[2], w[3]));
	// one atomic per block, and only where it would raise the maximum: those to
	// one address take 12 ns each.  Non-negative floats order as their bits.
	const unsigned b = __float_as_uint(m);
	if (threadIdx.x == 0 && b > __hip_atomic_load(out, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(out, b);
}

// A wave takes 16 rows of 32 columns at a time, a kilobyte of fragments in one
// store (lane l: row l % 16, columns 8 (l / 16) on), and a step along the rows.
// n = 9000, us: 173 -> 79 (6.3 TB/s), a row's eight columns per thread before.
template <typename E> __global__ __launch_bounds__(kB) void k_to_frag(const float *F, int ld, float s, E *out)
{
	typedef typename VecOf<E>::type V;
	const int lane = threadIdx.x & 63, nkb = ld >> 5;
	const unsigned blocks = (unsigned)(ld >> 4) * nkb, step = gridDim.x * (kB / 64);
	for (unsigned b = blockIdx.x * (kB / 64) + (threadIdx.x >> 6); b < blocks; b += step) {
		const unsigned row = b / nkb * 16 + (lane & 15), k = b % nkb * 32 + (lane >> 4) * 8;
		const float4 *f = (const float4 *)(F + (size_t)row * ld + k);
		const float4 a = f[0], c = f[1];
		V v;
		v[0] = (E)(a.x * s); v[1] = (E)(a.y * s); v[2] = (E)(a.z * s); v[3] = (E)(a.w * s);
		v[4] = (E)(c.x * s); v[5] = (E)(c.y * s); v[6] = (E)(c.z * s); v[7] = (E)(c.w * s);
		*(V *)(out + ((size_t)b * 64 + lane) * 8) = v;
	}
}

template <typename T> __global__ void k_fill(T *p, size_t count, T v)
{
	for (size_t i = blockIdx.x * (size_t)kB + threadIdx.x; i < count; i += (size_t)gridDim.x * kB) p[i] = v;
}

// What becomes of a low-precision product y = (A X)[i][c]: with y given, the
// product itself, y[i][c] = inv y.  Else one Jacobi sweep, v = rhs + rho o (inv
// y) and XTn <- v (fragment order); with rho_in (the adjoint's sweep v <- r +
// F^T (rho o v)) v = rhs + inv y and XTn <- rho o v.  Padding of XTn (rows >=
// nrhs, k >= n) is never written and stays zero.  With xT (the last sweep of a
// refinement) the FP64 iterate takes the correction, xT[c][i] += s v (first:
// xT[c][i] = s v), and wT (the adjoint's product input) becomes rho64 o xT.
template <typename E> struct SweepOut {
	int n, nrhs;
	float inv;
	bool rho_in, first;
	const float *rhs, *rho;
	E *XTn;
	double *xT, s, *wT;
	const double *rho64;
	float *y;

	// all but XTn: the next iterate's entry (0 where the product is asked for)
	__device__ __forceinline__ E value(int i, int c, int ld, float sum) const
	{
		const size_t t = (size_t)i * nrhs + c;
		if (y) {
			y[t] = sum * inv;
			return (E)0.f;
		}
		const float v = rho_in ? rhs[t] + sum * inv : rhs[t] + rho[t] * (sum * inv);
		if (xT) {
			const size_t q = (size_t)c * ld + i;
			const double x = (first ? 0.0 : xT[q]) + s * (double)v;
			xT[q] = x;
			if (wT) wT[q] = rho64[t] * x;
		}
		return (E)(rho_in ? rho[t] * v : v);
	}
	__device__ __forceinline__ void put(int i, int c, int ld, float sum) const
	{
		const E v = value(i, c, ld, sum);
		if (!y) XTn[frag_index(c, i, ld)] = v;
	}
};

// One block's rows of a sweep (block blk of the matrix; red: kSweepWaves RT CT
// 64 entries of LDS).  A block is eight waves: 8 / S row groups of 16 RT rows,
// the K range of each split over S waves.  Each wave streams its A
// fragments (two register sets of two k-blocks, one loading while the other
// feeds the MFMAs; the index is clamped past the chunk's end, those k-blocks
// are not multiplied), the partial tiles meet in LDS and are summed in chunk
// order, and the block's threads finish their rows (SweepOut).  The next
// iterate goes to a second buffer, as other blocks still read this one.
// A is read without the non-temporal policy where it stays in the 256 MB
// last-level cache from sweep to sweep (cached).
// Bound by that cache or HBM: the split inside the block keeps every CU busy
// where a block per row group and a second kernel for the sweep's update left
// CUs idle and paid a launch (one column tile, us per sweep, before -> now:
// n = 1024 8.0 -> 3.2, 4096 12.5 -> 5.3, 6144 20 -> 12.5, 9216 39 -> 25.0,
// 20224 187 -> 137 (6.0 TB/s), 32768 313 -> 302 (7.1 TB/s)).
constexpr int kSweepWaves = 8;
template <typename E, int RT, int CT>
__device__ __forceinline__ void sweep_rows(const E *__restrict__ A, const E *__restrict__ XT, int ld, int S, bool cached,
                                           int blk, f4 *red, const SweepOut<E> &o)
{
	typedef typename VecOf<E>::type V;
	constexpr int U = 2;
	const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int WR = kSweepWaves / S, wr = w % WR, s = w / WR;
	const int nkb = ld >> 5, cnt = nkb / S, nrt = ld >> 4;  // ld is a multiple of 256: nkb of 8
	const int rt0 = (blk * WR + wr) * RT;
	const V *Ap[RT];
#pragma unroll
	for (int r = 0; r < RT; r++) Ap[r] = (const V *)A + ((size_t)min(rt0 + r, nrt - 1) * nkb + s * cnt) * 64 + lane;
	const V *Bp = (const V *)XT + (size_t)(s * cnt) * 64 + lane;
	f4 acc[RT][CT];
#pragma unroll
	for (int r = 0; r < RT; r++)
#pragma unroll
		for (int c = 0; c < CT; c++) acc[r][c] = f4{0.f, 0.f, 0.f, 0.f};
	V a[2][U][RT], b[2][U][CT];
	auto run = [&](auto nt) {
		auto load = [&](int p, int k0) {
#pragma unroll
			for (int u = 0; u < U; u++) {
				const size_t k = (size_t)min(k0 + u, cnt - 1);
#pragma unroll
				for (int r = 0; r < RT; r++) {
					if constexpr (decltype(nt)::value) a[p][u][r] = __builtin_nontemporal_load(Ap[r] + k * 64);
					else a[p][u][r] = Ap[r][k * 64];
				}
#pragma unroll
				for (int c = 0; c < CT; c++) b[p][u][c] = Bp[((size_t)c * nkb + k) * 64];
			}
		};
		auto mma = [&](int p, int k0) {
#pragma unroll
			for (int u = 0; u < U; u++)
				if (k0 + u < cnt) {
#pragma unroll
					for (int r = 0; r < RT; r++)
#pragma unroll
						for (int c = 0; c < CT; c++) acc[r][c] = mfma(a[p][u][r], b[p][u][c], acc[r][c]);
				}
		};
		load(0, 0);
		for (int k = 0; k < cnt; k += 2 * U) {
			load(1, k + U);
			mma(0, k);
			load(0, k + 2 * U);
			mma(1, k + U);
		}
	};
	if (cached) run(std::integral_constant<bool, false>{});
	else run(std::integral_constant<bool, true>{});
#pragma unroll
	for (int r = 0; r < RT; r++)
#pragma unroll
		for (int c = 0; c < CT; c++) red[(((s * WR + wr) * RT + r) * CT + c) * 64 + lane] = acc[r][c];
	__syncthreads();
	// element (row, column) of a 16 x 16 tile: lane 16 (row / 4) + column, value row % 4
	const float *rf = (const float *)red;
	const int rows = WR * RT * 16, row0 = blk * rows, part = WR * RT * CT * 256;
	for (int e = threadIdx.x; e < rows * o.nrhs; e += kSweepWaves * 64) {
		const int rl = e / o.nrhs, c = e - rl * o.nrhs;
		if (row0 + rl >= o.n) break;
		const float *q = rf + ((rl >> 4) * CT + (c >> 4)) * 256 + (((rl & 15) >> 2) * 16 + (c & 15)) * 4 + (rl & 3);
		float y = 0.f;
		for (int k = 0; k < S; k++) y += q[k * part];
		o.put(row0 + rl, c, ld, y);
	}
}

// One block's rows (block blk of the matrix) of the whole FP64 residual for NC
// <= 4 right-hand sides on the vector FP64 units, where a 16-column MFMA would spend 13 of its 16 columns on padding:
// out[i][c] = base[i][c] + rho[i][c] * (F w)[i][c] - xT[c][i] (base, rho and xT
// may be null: 0, 1 and 0) and, into st, the sum of squares and max |out|.
// A wave owns kFxRows rows; per step each lane takes 4 consecutive k of each
// row (one 16-byte load per row, the next step's loads in flight) against w
// staged through LDS in chunks of 1024 k, column-major, so that a lane's 4
// values are two 16-byte reads.  KS of the block's four waves share rows, each
// taking every KS-th step of 256 k: a block is 32 / KS rows.  The 64 lane
// partials of the 8 NC sums are combined by a reduce-scatter (the exchanges
// over lane bits 5, 4, 3 halve the set each time and leave lane l with row
// l >> 3), then the KS waves' in a fixed order.
// Bound by HBM: 6.0-6.6 TB/s from n = 8192 up, FP64 work about half of that.
// Against the form with one block size (32 rows), 32-way LDS conflicts, 4
// columns for any NC and a second kernel for the residual (3 columns, us,
// first kernel alone): n = 1024 10.8 -> 4.7, 4096 30.5 -> 16.6, 9216 88.7 ->
// 61.9, 20224 290 -> 247, 32768 696 -> 643.
constexpr int kFxRows = 8;
constexpr int kFxChunk = 1024;
template <int NC, int KS> struct FxShared {
	double xs[NC * kFxChunk];
	double red[KS][4 / KS * kFxRows * NC];
	double stat[8];
};
template <int NC, int KS>
__device__ __forceinline__ void fx64_rows(const float *__restrict__ F, const double *__restrict__ wT, int ld, int n,
                                          int blk, FxShared<NC, KS> &sh, const double *xT, const double *base,
                                          const double *rho, double *out, double *st)
{
	typedef float fv4 __attribute__((ext_vector_type(4)));
	typedef double dv2 __attribute__((ext_vector_type(2)));
	constexpr int ROWS = 4 / KS * kFxRows, STEPS = kFxChunk / 256;
	static_assert(kFxRows == 8 && ROWS * NC <= kB, "the reduce-scatter assumes 8 rows; one thread per result");
	double *xs = sh.xs, *stat = sh.stat;
	auto &red = sh.red;
	const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
	const int rg = w / KS, ks = w % KS;
	const float *Fr = F + (size_t)(blk * ROWS + rg * kFxRows) * ld + 4 * lane;
	const int ns = ld / 256;
	double v[kFxRows * NC];
#pragma unroll
	for (int i = 0; i < kFxRows * NC; i++) v[i] = 0.0;
	fv4 a[kFxRows], an[kFxRows];
#pragma unroll
	for (int r = 0; r < kFxRows; r++)
		a[r] = __builtin_nontemporal_load((const fv4 *)(Fr + (size_t)r * ld + min(ks, ns - 1) * 256));
	for (int s0 = 0; s0 < ns; s0 += STEPS) {
		const int cnt = min(STEPS, ns - s0);
		__syncthreads();  // the previous chunk's reads are done
		for (int i = threadIdx.x; i < cnt * 128; i += kB)
#pragma unroll
			for (int c = 0; c < NC; c++)
				*(dv2 *)(xs + c * kFxChunk + 2 * i) = *(const dv2 *)(wT + (size_t)c * ld + s0 * 256 + 2 * i);
		__syncthreads();
#pragma unroll 1
		for (int q = ks; q < cnt; q += KS) {
			const int sn = min(s0 + q + KS, ns - 1);  // clamped: the last load of a wave is not used
#pragma unroll
			for (int r = 0; r < kFxRows; r++)
				an[r] = __builtin_nontemporal_load((const fv4 *)(Fr + (size_t)r * ld + sn * 256));
			double x[NC][4];
#pragma unroll
			for (int c = 0; c < NC; c++)
#pragma unroll
				for (int j = 0; j < 4; j++) x[c][j] = xs[c * kFxChunk + q * 256 + 4 * lane + j];
#pragma unroll
			for (int j = 0; j < 4; j++)
#pragma unroll
				for (int r = 0; r < kFxRows; r++) {
					const double f = (double)a[r][j];
#pragma unroll
					for (int c = 0; c < NC; c++) v[r * NC + c] = __builtin_fma(f, x[c][j], v[r * NC + c]);
				}
#pragma unroll
			for (int r = 0; r < kFxRows; r++) a[r] = an[r];
		}
	}
#pragma unroll
	for (int half = kFxRows * NC / 2, bit = 32; bit >= 8; half >>= 1, bit >>= 1) {
		const bool upper = (lane & bit) != 0;
#pragma unroll
		for (int i = 0; i < half; i++) {
			const double lo = v[i], hi = v[half + i];
			v[i] = (upper ? hi : lo) + __shfl_xor(upper ? lo : hi, bit);
		}
	}
#pragma unroll
	for (int bit = 4; bit > 0; bit >>= 1)
#pragma unroll
		for (int c = 0; c < NC; c++) v[c] += __shfl_xor(v[c], bit);
	if ((lane & 7) == 0)
#pragma unroll
		for (int c = 0; c < NC; c++) red[ks][(rg * kFxRows + (lane >> 3)) * NC + c] = v[c];
	__syncthreads();
	double ss = 0.0, mx = 0.0;
	const int e = threadIdx.x, i = blk * ROWS + e / NC, c = e % NC;
	if (e < ROWS * NC && i < n) {
		double y = red[0][e];
#pragma unroll
		for (int k = 1; k < KS; k++) y += red[k][e];
		const size_t t = (size_t)i * NC + c;
		const double o = (base ? base[t] : 0.0) + (rho ? rho[t] : 1.0) * y - (xT ? xT[(size_t)c * ld + i] : 0.0);
		out[t] = o;
		ss = o * o;
		mx = fabs(o);
	}
	for (int off = 32; off > 0; off >>= 1) {
		ss += __shfl_xor(ss, off);
		mx = fmax(mx, __shfl_xor(mx, off));
	}
	if (lane == 0) {
		stat[2 * w] = ss;
		stat[2 * w + 1] = mx;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		st[0] = stat[0] + stat[2] + stat[4] + stat[6];
		st[1] = fmax(fmax(stat[1], stat[3]), fmax(stat[5], stat[7]));
	}
}

// the matrix's 16-bit copy stays in the 256 MB last-level cache between
// sweeps: up to 11.5k rows (us per sweep, cached against non-temporal: n = 4096
// 5.3, 8.0; 9216 25.0, 37.1; 12288 48.9, 50.6; 16384 95.6, 82.9; 20224 144.5,
// 136.5)
bool stays_cached(size_t elements) { return 2 * elements <= (size_t)256 << 20; }

#define HIP_OK(expr, what)                                          \
	do {                                                            \
		hipError_t e_ = (expr);                                     \
		if (e_ != hipSuccess) {                                     \
			err = std::string(what) + ": " + hipGetErrorString(e_); \
			return -1;                                              \
		}                                                           \
	} while (0)

template <typename T> struct Buf {
	T *p = nullptr;
	size_t n = 0;
	Buf() = default;
	Buf(const Buf &) = delete;
	Buf &operator=(const Buf &) = delete;
	~Buf()
	{
		if (p) (void)hipFree(p);
	}
	int alloc(size_t count, std::string &err)
	{
		if (count <= n && p) return 0;
		if (p) (void)hipFree(p);
		p = nullptr;
		n = 0;
		if (count == 0) return 0;
		HIP_OK(hipMalloc(&p, count * sizeof(T)), "hipMalloc");
		n = count;
		return 0;
	}
};

int grid_for(size_t total) { return (int)std::min<size_t>((total + kB - 1) / kB, 8192); }

double ms_since(std::chrono::steady_clock::time_point a)
{
	return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - a).count();
}


