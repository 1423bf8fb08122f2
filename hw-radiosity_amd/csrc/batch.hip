// Batched mixed-precision gather over scenes of uneven size (see batch.h).
//
// HBM layout (scene s, n_s patches, ld_s = n_s rounded up to 256):
//   F32   ld_s^2 floats at off[s], row-major (the matrix of record)
//   F16 / BF16  ld_s^2 at off[s], MFMA fragment order, one power-of-two scale
//         for the whole batch (FP16)
//   rows  n_s * 3 at voff[s]: rho, E, residual, scaled residual, answer
//   xT    16 x ld_s at xoff[s]: FP64 iterate (rows 0..2 used), and its
//         low-precision copies (two, read and written in turn) in fragment
//         order for the MFMA B operand
// Work lists, sorted by scene: residual tiles {scene, block of 32 / KS rows};
// sweep tiles {scene, block of 16 rt 8 / S rows, S}, whose shape goes by the
// schedule; element tiles {scene, first element} of 256 elements, never
// straddling a scene, so that per-scene norms are sums over a fixed range of
// tile statistics.
#include "batch.h"
#include "linear.h"

#include "pack.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

namespace rgpu {
namespace {

#include "lin_common.h"
#include "stage.h"

constexpr int NR = 3;           // right-hand sides per scene (RGB)
constexpr int kPersist = 4096;  // blocks of the element-walking kernels

struct BMeta {
	int n, ld;
	long long off, voff, xoff;
};

// one sweep of every active scene: block after block of the list (sweep_rows)
// in a persistent grid
template <typename E, int RT>
__global__ __launch_bounds__(kSweepWaves * 64) void k_bsweep(const int4 *tiles, int t0, int t1, const BMeta *meta,
                                                             const int *active, const E *F, const E *X, bool cached,
                                                             float inv, const float *r32, const float *rho, E *Xn,
                                                             double *xT, const double *scale)
{
	__shared__ f4 red[kSweepWaves * RT * 64];
	for (int t = t0 + blockIdx.x; t < t1; t += gridDim.x) {
		const int4 tl = tiles[t];  // scene, block, S
		if (!active[tl.x]) continue;
		const BMeta m = meta[tl.x];
		SweepOut<E> o{};
		o.n = m.n, o.nrhs = NR, o.inv = inv, o.rhs = r32 + m.voff, o.rho = rho + m.voff, o.XTn = Xn + m.xoff;
		if (xT) o.xT = xT + m.xoff, o.s = scale[tl.x];
		sweep_rows<E, RT, 1>(F + m.off, X + m.xoff, m.ld, tl.z, cached, tl.y, red, o);
		__syncthreads();  // red is read to the end
	}
}

// FP64 residual r = E + rho o (F x) - x of every active scene, with the norms
// of each tile
template <int KS>
__global__ __launch_bounds__(kB) void k_bfx(const int2 *tiles, int t0, int t1, const BMeta *meta, const int *active,
                                            const float *__restrict__ F32, const double *xT, const double *E,
                                            const double *rho, double *r, double *blk)
{
	__shared__ FxShared<NR, KS> sh;
	for (int t = t0 + blockIdx.x; t < t1; t += gridDim.x) {
		const int2 tl = tiles[t];
		if (!active[tl.x]) continue;
		const BMeta m = meta[tl.x];
		const double *x = xT + m.xoff;
		fx64_rows<NR, KS>(F32 + m.off, x, m.ld, m.n, tl.y, sh, x, E + m.voff, rho + m.voff, r + m.voff, blk + 2 * t);
		__syncthreads();
	}
}

// the first residual (x = 0): r = E, rho in FP32, and each element tile's norms
__global__ __launch_bounds__(kB) void k_binit(const int2 *etiles, int e0, int e1, const BMeta *meta, const double *E,
                                              const double *rho, double *r, float *rho32, double *blk)
{
	__shared__ double red[8];
	for (int t = e0 + blockIdx.x; t < e1; t += gridDim.x) {
		const int2 et = etiles[t];
		const BMeta m = meta[et.x];
		const int idx = et.y + threadIdx.x;
		double ss = 0.0, mx = 0.0;
		if (idx < m.n * NR) {
			const size_t g = m.voff + idx;
			const double v = E[g];
			r[g] = v;
			rho32[g] = (float)rho[g];
			ss = v * v;
			mx = fabs(v);
		}
		for (int off = 32; off > 0; off >>= 1) {
			ss += __shfl_xor(ss, off);
			mx = fmax(mx, __shfl_xor(mx, off));
		}
		if ((threadIdx.x & 63) == 0) {
			red[2 * (threadIdx.x >> 6)] = ss;
			red[2 * (threadIdx.x >> 6) + 1] = mx;
		}
		__syncthreads();
		if (threadIdx.x == 0) {
			blk[2 * t] = red[0] + red[2] + red[4] + red[6];
			blk[2 * t + 1] = fmax(fmax(red[1], red[3]), fmax(red[5], red[7]));
		}
		__syncthreads();
	}
}

// per scene (one wave each): norms from its tiles [tb, te) in a fixed order;
// relative residual, scale for the next correction, still active?  state (host
// memory): the residual and the flag for the host's own look
struct BState {
	double rel;
	int active, pad;
};
__global__ void k_bnorm(int sc0, const int *tb, const int *te, const double *blk, int *active, double *enorm,
                        double *scale, BState *state, double tol, int first)
{
	const int s = sc0 + blockIdx.x;
	if (!active[s]) return;
	double ss = 0.0, mx = 0.0;
	for (int t = tb[s] + threadIdx.x; t < te[s]; t += 64) {
		ss += blk[2 * t];
		mx = fmax(mx, blk[2 * t + 1]);
	}
	for (int off = 32; off > 0; off >>= 1) {
		ss += __shfl_xor(ss, off);
		mx = fmax(mx, __shfl_xor(mx, off));
	}
	if (threadIdx.x != 0) return;
	const double e = first ? sqrt(ss) : enorm[s];
	if (first) enorm[s] = e;
	const double r = e > 0.0 ? sqrt(ss) / e : 0.0;
	const int act = (r > tol && mx > 0.0) ? 1 : 0;
	scale[s] = mx;
	active[s] = act;
	state[s].rel = r;
	state[s].active = act;
}

// r32 = r / scale; XT <- r32 (fragment order)
template <typename E>
__global__ __launch_bounds__(kB) void k_bscale(const int2 *etiles, int e0, int e1, const BMeta *meta,
                                               const int *active, const double *r, const double *scale, float *r32,
                                               E *XT)
{
	for (int t = e0 + blockIdx.x; t < e1; t += gridDim.x) {
		const int2 et = etiles[t];
		if (!active[et.x]) continue;
		const BMeta m = meta[et.x];
		const int idx = et.y + threadIdx.x;
		if (idx >= m.n * NR) continue;
		const size_t g = m.voff + idx;
		const float v = (float)(r[g] / scale[et.x]);
		r32[g] = v;
		XT[m.xoff + frag_index(idx % NR, idx / NR, m.ld)] = (E)v;
	}
}

// out = x, the scenes' rows in the caller's order
__global__ __launch_bounds__(kB) void k_brows(const int2 *etiles, int ne, const BMeta *meta, const double *xT, double *out)
{
	for (int t = blockIdx.x; t < ne; t += gridDim.x) {
		const int2 et = etiles[t];
		const BMeta m = meta[et.x];
		const int idx = et.y + threadIdx.x;
		if (idx < m.n * NR) out[m.voff + idx] = xT[m.xoff + (size_t)(idx % NR) * m.ld + idx / NR];
	}
}

}  // namespace

struct SceneBatch::Impl {
	int count = 0;
	std::vector<int> n, ld, tb, te, gtb, gte, etb, ete;
	std::vector<BMeta> meta;
	size_t fsize = 0, vsize = 0, xsize = 0;
	int ntiles = 0, ngtiles = 0, netiles = 0, total = 0;
	int ks = 4;             // waves per row group of the residual (32 / ks rows a tile)
	BatchTile gs{0, -1, 0}; // current sweep schedule; kc = 0: S = 8 whatever the size
	BatchTile best[2] = {{0, 0, 0}, {0, 0, 0}};  // autotuned, per precision
	bool forced = false;    // set_tile overrides the autotuner
	hipStream_t st = nullptr;
	hipEvent_t e0 = nullptr, e1 = nullptr;
	Stage stage;
	Buf<double> out;  // the answer as the caller takes it
	Buf<float> F32, r32, rho32;
	Buf<_Float16> F16, X16[2];
	Buf<__bf16> FB, XB[2];
	Buf<double> E64, rho64, r64, xT, blk, enorm, scale;
	Buf<int> active, d_tb, d_te, d_etb, d_ete;
	Buf<int4> gtiles;
	Buf<int2> tiles, etiles;
	Buf<BMeta> d_meta;
	Buf<unsigned> umax;
	bool have16 = false, haveb = false;
	float s16 = 1.f;
	// captured once and replayed: the start (clears, first norms) and one
	// refinement
	hipGraphExec_t exec[2] = {};
	hipGraph_t graph[2] = {};
	int g_prec = -1, g_sweeps = -1, g_nodes[2] = {};
	double g_tol = -1.0;

	void drop_graph()
	{
		for (int k = 0; k < 2; k++) {
			if (exec[k]) (void)hipGraphExecDestroy(exec[k]);
			if (graph[k]) (void)hipGraphDestroy(graph[k]);
			exec[k] = nullptr;
			graph[k] = nullptr;
		}
		g_prec = -1;
	}
	BState *state() { return reinterpret_cast<BState *>(stage.stats); }
	int ensure_lowp(int prec, std::string &err)
	{
		if ((prec == PREC_F16 && have16) || (prec == PREC_BF16 && haveb)) return 0;
		// a captured graph bakes in the FP16 scale (its sweeps multiply by
		// 1/s16) and reads the copy being rebuilt: capture again
		drop_graph();
		if (prec == PREC_F16) {
			if (umax.alloc(1, err) || F16.alloc(fsize, err)) return -1;
			hipLaunchKernelGGL(k_fill<unsigned>, dim3(1), dim3(kB), 0, st, umax.p, (size_t)1, 0u);
			hipLaunchKernelGGL(k_absmax, dim3(4096), dim3(kB), 0, st, F32.p, fsize, umax.p);
			unsigned bits = 0;
			HIP_OK(hipMemcpyAsync(&bits, umax.p, 4, hipMemcpyDeviceToHost, st), "absmax");
			HIP_OK(hipStreamSynchronize(st), "absmax");
			float m;
			std::memcpy(&m, &bits, 4);
			if (!std::isfinite(m)) {
				err = "matrix has non-finite entries";
				return -1;
			}
			int e = 0;
			if (m > 0.f) e = std::max(-60, std::min(60, (int)std::floor(std::log2(16384.0 / m))));
			s16 = std::ldexp(1.0f, e);
			for (int s = 0; s < count; s++)
				hipLaunchKernelGGL(k_to_frag<_Float16>, dim3(2048), dim3(kB), 0, st, F32.p + meta[s].off, ld[s], s16,
				                   F16.p + meta[s].off);
			have16 = true;
		} else {
			if (FB.alloc(fsize, err)) return -1;
			for (int s = 0; s < count; s++)
				hipLaunchKernelGGL(k_to_frag<__bf16>, dim3(2048), dim3(kB), 0, st, F32.p + meta[s].off, ld[s], 1.0f,
				                   FB.p + meta[s].off);
			haveb = true;
		}
		HIP_OK(hipGetLastError(), "convert");
		return 0;
	}

	// the default schedule: every wave of a block on the same rows, 16 of them,
	// 32 from four blocks of 16 per CU up, 64 from sixty-four (ms per solve at 16,
	// 32, 64: 8 rooms of 500 to 1000 patches 0.312, 0.305, 0.332; 48 of 500 to
	// 4000 2.45, 2.26, 2.27; 64 of 3000 to 8000 22.5, 20.5, 20.1)
	BatchTile rule() const
	{
		size_t rows = 0;
		for (int l : ld) rows += l;
		return BatchTile{rows / 16 < 1024 ? 1 : rows / 16 < 16384 ? 2 : 4, 0, 16384};
	}
	static bool valid_tile(const BatchTile &g)
	{
		return (g.rt == 1 || g.rt == 2 || g.rt == 4) &&
		       (g.kc == 1024 || g.kc == 2048 || g.kc == 4096 || g.kc == 8192) && g.grid >= 64 && g.grid <= 16384;
	}
	// rebuilds the sweep's tile list for schedule g (g.kc = 0: rule())
	int set_sched(const BatchTile &g, std::string &err)
	{
		if (g.kc != 0 && !valid_tile(g)) {
			err = "batch tile: rt in {1, 2, 4}, kc in {1024, 2048, 4096, 8192}, grid 64..16384";
			return -1;
		}
		if (g.rt == gs.rt && g.kc == gs.kc && g.grid == gs.grid) return 0;
		// largest scenes first: the blocks that take the longest tiles start
		// first, which shortens the tail of a launch over the whole batch
		std::vector<int> ord(count);
		for (int s = 0; s < count; s++) ord[s] = s;
		std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return ld[a] > ld[b]; });
		std::vector<int4> tl;
		gtb.assign(count, 0);
		gte.assign(count, 0);
		for (const int s : ord) {
			int S = kSweepWaves;  // K split: the largest power of two up to 8 and ld / kc rounded up
			while (g.kc && S > 1 && (S - 1) * g.kc >= ld[s]) S /= 2;
			gtb[s] = (int)tl.size();
			const int wr = kSweepWaves / S * g.rt;  // row tiles per block
			for (int b = 0; b < (ld[s] / 16 + wr - 1) / wr; b++) tl.push_back(make_int4(s, b, S, 0));
			gte[s] = (int)tl.size();
		}
		ngtiles = (int)tl.size();
		HIP_OK(hipStreamSynchronize(st), "batch tile");
		if (gtiles.alloc(tl.size(), err)) return -1;
		HIP_OK(hipMemcpyAsync(gtiles.p, tl.data(), tl.size() * sizeof(int4), hipMemcpyHostToDevice, st), "batch tile");
		HIP_OK(hipStreamSynchronize(st), "batch tile");
		gs = g;
		drop_graph();
		return 0;
	}
	// one sweep over tiles [g0, g1); last: it adds the correction to x
	template <typename E> void sweep(const E *F, const E *X, E *Xn, int g0, int g1, float inv, bool last)
	{
		const dim3 grid(std::max(1, std::min(gs.grid, g1 - g0))), blk(kSweepWaves * 64);
		const bool cached = stays_cached(fsize);
		double *x = last ? xT.p : nullptr;
#define G(R)                                                                                                           \
	hipLaunchKernelGGL((k_bsweep<E, R>), grid, blk, 0, st, gtiles.p, g0, g1, d_meta.p, active.p, F, X, cached, inv,     \
	                   r32.p, rho32.p, Xn, x, scale.p)
		if (gs.rt == 1) G(1);
		else if (gs.rt == 2) G(2);
		else G(4);
#undef G
	}
	// times one sweep (every scene active) for each candidate schedule on this
	// batch's matrices and keeps the fastest
	template <typename E> int tune(const E *Fl, Buf<E> (&X)[2], float inv, BatchTile &out, std::string &err)
	{
		const size_t V = vsize;
		hipLaunchKernelGGL(k_fill<int>, dim3(grid_for((size_t)count)), dim3(kB), 0, st, active.p, (size_t)count, 1);
		hipLaunchKernelGGL(k_fill<float>, dim3(grid_for(V)), dim3(kB), 0, st, r32.p, V, 0.f);
		hipLaunchKernelGGL(k_fill<float>, dim3(grid_for(V)), dim3(kB), 0, st, rho32.p, V, 0.f);
		HIP_OK(hipGetLastError(), "tune");
		double best_ms = 1e300;
		BatchTile pick = gs;
		for (int rt : {1, 2, 4})
			for (int kc : {1024, 2048, 4096, 8192})
				for (int grid : {512, 1024, 2048, 4096}) {
					if (set_sched(BatchTile{rt, kc, grid}, err)) return -1;
					constexpr int kReps = 3;
					for (int r = 0; r <= kReps; r++) {
						if (r == 1) HIP_OK(hipEventRecord(e0, st), "tune");
						sweep<E>(Fl, X[0].p, X[1].p, 0, ngtiles, inv, false);
					}
					HIP_OK(hipEventRecord(e1, st), "tune");
					HIP_OK(hipEventSynchronize(e1), "tune");
					float ms = 0.f;
					HIP_OK(hipEventElapsedTime(&ms, e0, e1), "tune");
					if (ms < best_ms) {
						best_ms = ms;
						pick = gs;
					}
				}
		out = pick;
		return set_sched(pick, err);
	}
	// the iterate's two buffers: padding zero, never written
	template <typename E> int iterates(Buf<E> (&X)[2], std::string &err)
	{
		for (Buf<E> &x : X)
			if (!x.p) {
				if (x.alloc(xsize, err)) return -1;
				hipLaunchKernelGGL(k_fill<E>, dim3(grid_for(xsize)), dim3(kB), 0, st, x.p, xsize, (E)0.f);
			}
		return 0;
	}

	// The solve's kernels for scenes [sc0, sc1) (one scene, or all: the sweep
	// list is in its own scene order); both return the number of launches.
	// start: x = 0, the first residual and its norms
	int start(int sc0, int sc1, double tol)
	{
		const int q0 = etb[sc0], q1 = ete[sc1 - 1];
		hipLaunchKernelGGL(k_binit, dim3(std::max(1, std::min(kPersist, q1 - q0))), dim3(kB), 0, st, etiles.p, q0, q1,
		                   d_meta.p, E64.p, rho64.p, r64.p, rho32.p, blk.p);
		hipLaunchKernelGGL(k_bnorm, dim3(sc1 - sc0), dim3(64), 0, st, sc0, d_etb.p, d_ete.p, blk.p, active.p, enorm.p,
		                   scale.p, state(), tol, 1);
		return 2;
	}
	// one refinement: the scaled residual, sweeps, the new residual and norms
	template <typename E> int refine(const E *F, Buf<E> (&X)[2], int sc0, int sc1, int sweeps, double tol, float inv)
	{
		const int t0 = tb[sc0], t1 = te[sc1 - 1], q0 = etb[sc0], q1 = ete[sc1 - 1];
		const bool all = sc0 == 0 && sc1 == count;
		const int g0 = all ? 0 : gtb[sc0], g1 = all ? ngtiles : gte[sc0];  // else sc1 = sc0 + 1
		hipLaunchKernelGGL(k_bscale<E>, dim3(std::max(1, std::min(kPersist, q1 - q0))), dim3(kB), 0, st, etiles.p, q0, q1,
		                   d_meta.p, active.p, r64.p, scale.p, r32.p, X[0].p);
		for (int m = 0; m < sweeps; m++) sweep<E>(F, X[m & 1].p, X[(m + 1) & 1].p, g0, g1, inv, m == sweeps - 1);
		const dim3 gt(t1 - t0);
		if (ks == 1)
			hipLaunchKernelGGL(k_bfx<1>, gt, dim3(kB), 0, st, tiles.p, t0, t1, d_meta.p, active.p, F32.p, xT.p, E64.p,
			                   rho64.p, r64.p, blk.p);
		else
			hipLaunchKernelGGL(k_bfx<4>, gt, dim3(kB), 0, st, tiles.p, t0, t1, d_meta.p, active.p, F32.p, xT.p, E64.p,
			                   rho64.p, r64.p, blk.p);
		hipLaunchKernelGGL(k_bnorm, dim3(sc1 - sc0), dim3(64), 0, st, sc0, d_tb.p, d_te.p, blk.p, active.p, enorm.p,
		                   scale.p, state(), tol, 0);
		return 3 + sweeps;
	}
	int clears()
	{
		hipLaunchKernelGGL(k_fill<double>, dim3(grid_for(xsize)), dim3(kB), 0, st, xT.p, xsize, 0.0);
		hipLaunchKernelGGL(k_fill<int>, dim3(grid_for((size_t)count)), dim3(kB), 0, st, active.p, (size_t)count, 1);
		return 2;
	}
	// what record launches, as graph k
	template <typename L> int capture(int k, L record, std::string &err)
	{
		HIP_OK(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), "capture");
		const int l = record();
		hipGraph_t g = nullptr;
		const hipError_t ce = hipStreamEndCapture(st, &g);
		if (ce != hipSuccess || !g) {
			err = std::string("graph capture: ") + hipGetErrorString(ce);
			return -1;
		}
		graph[k] = g;
		HIP_OK(hipGraphInstantiate(&exec[k], graph[k], nullptr, nullptr, 0), "graph instantiate");
		g_nodes[k] = l;
		return 0;
	}
	// the whole solve; launches and graph build time out
	template <typename E>
	int run(const E *F, Buf<E> (&X)[2], int prec, bool use_graph, int outer, int sweeps, double tol, float inv,
	        int &launches, double &build_ms, std::string &err)
	{
		if (!use_graph) {  // scene after scene
			HIP_OK(hipEventRecord(e0, st), "event");
			launches += clears();
			for (int s = 0; s < count; s++) {
				launches += start(s, s + 1, tol);
				for (int o = 0; o < outer; o++) launches += refine<E>(F, X, s, s + 1, sweeps, tol, inv);
			}
			HIP_OK(hipEventRecord(e1, st), "event");
			return 0;
		}
		if (!(exec[0] && exec[1] && g_prec == prec && g_sweeps == sweeps && g_tol == tol)) {
			drop_graph();
			const auto c0 = std::chrono::steady_clock::now();
			if (capture(0, [&] { return clears() + start(0, count, tol); }, err) ||
			    capture(1, [&] { return refine<E>(F, X, 0, count, sweeps, tol, inv); }, err)) {
				drop_graph();
				return -1;
			}
			g_prec = prec;
			g_sweeps = sweeps;
			g_tol = tol;
			build_ms = ms_since(c0);
		}
		HIP_OK(hipEventRecord(e0, st), "event");
		HIP_OK(hipGraphLaunch(exec[0], st), "graph launch");
		launches += g_nodes[0];
		for (int o = 0; o < outer; o++) {
			// a graph launch per refinement, until no scene is above tol
			HIP_OK(hipStreamSynchronize(st), "batch solve");
			bool any = false;
			for (int s = 0; s < count && !any; s++) any = state()[s].active != 0;
			if (!any) break;
			HIP_OK(hipGraphLaunch(exec[1], st), "graph launch");
			launches += g_nodes[1];
		}
		HIP_OK(hipEventRecord(e1, st), "event");
		return 0;
	}
};

SceneBatch::~SceneBatch()
{
	if (!d_) return;
	if (d_->st) (void)hipStreamSynchronize(d_->st);
	d_->drop_graph();
	if (d_->e0) (void)hipEventDestroy(d_->e0);
	if (d_->e1) (void)hipEventDestroy(d_->e1);
	hipStream_t s = d_->st;
	delete d_;
	if (s) (void)hipStreamDestroy(s);
}

SceneBatch *SceneBatch::create(int count, const int *n, std::string &err)
{
	if (count <= 0 || count > 65536 || !n) {
		err = "batch: count must be 1..65536";
		return nullptr;
	}
	for (int s = 0; s < count; s++)
		if (n[s] <= 0 || n[s] > 65536) {
			err = "batch: scene sizes must be 1..65536";
			return nullptr;
		}
	int ndev = 0;
	if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
		err = "no HIP device available";
		return nullptr;
	}
	SceneBatch *B = new SceneBatch();
	B->d_ = new Impl();
	Impl &d = *B->d_;
	d.count = count;
	size_t rows = 0;
	for (int s = 0; s < count; s++) rows += (n[s] + 255) / 256 * 256;
	// residual rows per tile: 32, or 8 while that leaves CUs without a block (ms
	// per solve at 32 and 8: 20 rooms of 500 to 2000 patches 0.508, 0.548; 48 of
	// 500 to 4000 2.12, 2.26; 8 of 500 to 1000 0.306, 0.305)
	d.ks = rows / 32 < 256 ? 4 : 1;
	std::vector<int2> tl, el;
	for (int s = 0; s < count; s++) {
		BMeta m;
		m.n = n[s];
		m.ld = (n[s] + 255) / 256 * 256;
		m.off = (long long)d.fsize;
		m.voff = (long long)d.vsize;
		m.xoff = (long long)d.xsize;
		d.fsize += (size_t)m.ld * m.ld;
		d.vsize += (size_t)m.n * NR;
		d.xsize += (size_t)16 * m.ld;
		d.n.push_back(m.n);
		d.ld.push_back(m.ld);
		d.meta.push_back(m);
		d.tb.push_back((int)tl.size());
		for (int b = 0; b < m.ld / 32 * d.ks; b++) tl.push_back(make_int2(s, b));
		d.te.push_back((int)tl.size());
		d.etb.push_back((int)el.size());
		for (int e = 0; e < m.n * NR; e += kB) el.push_back(make_int2(s, e));
		d.ete.push_back((int)el.size());
		d.total += m.n;
	}
	d.ntiles = (int)tl.size();
	d.netiles = (int)el.size();
	std::string e;
	if (hipStreamCreateWithFlags(&d.st, hipStreamNonBlocking) != hipSuccess || hipEventCreate(&d.e0) != hipSuccess ||
	    hipEventCreate(&d.e1) != hipSuccess) {
		err = "stream/event creation failed";
		delete B;
		return nullptr;
	}
	const size_t V = d.vsize;
	if (d.F32.alloc(d.fsize, e) || d.r32.alloc(V, e) || d.rho32.alloc(V, e) || d.E64.alloc(V, e) ||
	    d.rho64.alloc(V, e) || d.r64.alloc(V, e) || d.out.alloc(V, e) || d.stage.init(e) ||
	    d.stage.stat_room((size_t)count * (sizeof(BState) / sizeof(double)), e) || d.xT.alloc(d.xsize, e) ||
	    d.blk.alloc((size_t)std::max(d.netiles, d.ntiles) * 2, e) || d.enorm.alloc(count, e) || d.scale.alloc(count, e) ||
	    d.active.alloc(count, e) || d.d_tb.alloc(count, e) || d.d_te.alloc(count, e) || d.d_etb.alloc(count, e) ||
	    d.d_ete.alloc(count, e) || d.tiles.alloc(tl.size(), e) || d.etiles.alloc(el.size(), e) ||
	    d.d_meta.alloc(count, e)) {
		err = e;
		delete B;
		return nullptr;
	}
	if (hipMemsetAsync(d.F32.p, 0, d.fsize * 4, d.st) != hipSuccess ||
	    hipMemcpyAsync(d.tiles.p, tl.data(), tl.size() * sizeof(int2), hipMemcpyHostToDevice, d.st) != hipSuccess ||
	    hipMemcpyAsync(d.etiles.p, el.data(), el.size() * sizeof(int2), hipMemcpyHostToDevice, d.st) != hipSuccess ||
	    hipMemcpyAsync(d.d_meta.p, d.meta.data(), count * sizeof(BMeta), hipMemcpyHostToDevice, d.st) != hipSuccess ||
	    hipMemcpyAsync(d.d_tb.p, d.tb.data(), count * 4, hipMemcpyHostToDevice, d.st) != hipSuccess ||
	    hipMemcpyAsync(d.d_te.p, d.te.data(), count * 4, hipMemcpyHostToDevice, d.st) != hipSuccess ||
	    hipMemcpyAsync(d.d_etb.p, d.etb.data(), count * 4, hipMemcpyHostToDevice, d.st) != hipSuccess ||
	    hipMemcpyAsync(d.d_ete.p, d.ete.data(), count * 4, hipMemcpyHostToDevice, d.st) != hipSuccess ||
	    hipStreamSynchronize(d.st) != hipSuccess) {
		err = "batch upload failed";
		delete B;
		return nullptr;
	}
	if (d.set_sched(d.rule(), err)) {
		delete B;
		return nullptr;
	}
	return B;
}

int SceneBatch::count() const { return d_->count; }
int SceneBatch::n(int s) const { return d_->n[s]; }
int SceneBatch::ld(int s) const { return d_->ld[s]; }
int SceneBatch::total() const { return d_->total; }

float *SceneBatch::matrix32(int s)
{
	d_->have16 = d_->haveb = false;
	return d_->F32.p + d_->meta[s].off;
}

int SceneBatch::set_matrix(int s, const float *F, std::string &err)
{
	if (s < 0 || s >= d_->count) {
		err = "batch: scene index out of range";
		return -1;
	}
	const int n = d_->n[s], ld = d_->ld[s];
	HIP_OK(hipMemcpy2D(matrix32(s), (size_t)ld * 4, F, (size_t)n * 4, (size_t)n * 4, n, hipMemcpyHostToDevice),
	       "set matrix");
	return 0;
}

int SceneBatch::autotune(int prec, BatchTile &out, std::string &err)
{
	Impl &d = *d_;
	if (prec != PREC_F16 && prec != PREC_BF16) {
		err = "batch: precision must be FP16 or BF16";
		return -1;
	}
	if (d.ensure_lowp(prec, err)) return -1;
	const int pi = prec == PREC_F16 ? 0 : 1;
	if (prec == PREC_F16) {
		if (d.iterates(d.X16, err) || d.tune<_Float16>(d.F16.p, d.X16, 1.0f / d.s16, d.best[pi], err)) return -1;
	} else {
		if (d.iterates(d.XB, err) || d.tune<__bf16>(d.FB.p, d.XB, 1.0f, d.best[pi], err)) return -1;
	}
	d.forced = false;
	out = d.best[pi];
	return 0;
}

int SceneBatch::set_tile(const BatchTile &t, std::string &err)
{
	if (d_->set_sched(t, err)) return -1;
	d_->forced = true;
	return 0;
}

int SceneBatch::solve(int prec, bool graph, const double *rho, const double *E, double tol, int outer, int sweeps,
                      double *Bout, double *rel_res, double *info, std::string &err)
{
	Impl &d = *d_;
	if (prec != PREC_F16 && prec != PREC_BF16) {
		err = "batch: precision must be FP16 or BF16";
		return -1;
	}
	if (outer < 0 || outer > 64 || sweeps <= 0 || sweeps > 64) {
		err = "batch: outer must be 0..64 and sweeps 1..64";
		return -1;
	}
	if (d.ensure_lowp(prec, err)) return -1;
	if (!d.forced) {  // the tuned schedule, or the rule's
		const BatchTile &b = d.best[prec == PREC_F16 ? 0 : 1];
		if (d.set_sched(b.rt == 0 ? d.rule() : b, err)) return -1;
	}
	const size_t V = d.vsize;
	HIP_OK(hipStreamSynchronize(d.st), "batch solve");  // nothing of an earlier call is in flight
	d.stage.begin();
	if (d.stage.up(d.rho64.p, rho, V * 8, d.st, err) || d.stage.up(d.E64.p, E, V * 8, d.st, err)) return -1;
	const float inv = prec == PREC_F16 ? 1.0f / d.s16 : 1.0f;
	double build_ms = 0.0;
	int launches = 0;
	if (prec == PREC_F16 ? d.iterates(d.X16, err) || d.run<_Float16>(d.F16.p, d.X16, prec, graph, outer, sweeps, tol, inv,
	                                                                 launches, build_ms, err)
	                     : d.iterates(d.XB, err) || d.run<__bf16>(d.FB.p, d.XB, prec, graph, outer, sweeps, tol, inv,
	                                                              launches, build_ms, err))
		return -1;
	hipLaunchKernelGGL(k_brows, dim3(std::max(1, std::min(kPersist * 4, d.netiles))), dim3(kB), 0, d.st, d.etiles.p,
	                   d.netiles, d.d_meta.p, d.xT.p, d.out.p);
	HIP_OK(hipGetLastError(), "batch launch");
	if (d.stage.down(Bout, d.out.p, V * 8, d.st, err)) return -1;
	float ms = 0.f;
	HIP_OK(hipEventElapsedTime(&ms, d.e0, d.e1), "event");
	int above = 0;
	for (int s = 0; s < d.count; s++) {
		rel_res[s] = d.state()[s].rel;
		above += d.state()[s].active;
	}
	if (info) {
		info[0] = ms;
		info[1] = build_ms;
		info[2] = launches;
		info[3] = above;
	}
	return 0;
}

}  // namespace rgpu
