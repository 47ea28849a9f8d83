/* sgs_patch.hip -- several sweeps of multicolour symmetric Gauss-Seidel per launch, on
 * overlapping patches of the cell graph.
 *
 * An application of `sweeps` symmetric sweeps is a chain of 2 sweeps (colours - 1) + 1 colour
 * passes: 0, 1, .., C-1, C-2, .., 0, 1, .., each pass replacing the cells of its colour by
 * D_i^-1 (r_i - sum_j A_ij z_j). One launch per pass (k_sgs_rec, linalg.hip) is bound by launches
 * on small meshes (4.5 us a pass on 98,304 cells, 3.3 us on 4,608) and by re-reading the factors
 * in every pass on large ones. Here a workgroup owns a compact patch of cells, loads the patch
 * and a rim around it, performs the passes of up to four sweeps on its copy and writes the
 * patch's own cells: with each pass the part of the copy that still has the value the
 * colour-by-colour chain gives shrinks by one ring of cells, and the rim is as wide as that
 * takes. The rim's cells are computed by several workgroups, all with the same result, so the
 * outcome equals the colour passes bit for bit; there is no communication between workgroups.
 *
 * On the way down the colours, cells of a colour 0 < c < C-1 are computed only where a neighbour
 * has a higher colour: the others' neighbours have not changed since the way up, so the pass
 * would repeat their values (with 3 colours, the third holding 0.4% of the cells, a third of all
 * cell updates).
 *
 * The iterates between two launches alternate between the result and a scratch vector, because
 * other workgroups still read the rim's old values while one writes its cells.
 */
#include "fvx_internal.hpp"
#include "wave.hpp"
#include "blocks.hpp"
#include "threads.hpp"
#include <algorithm>
#include <atomic>
#include <cmath>
#include <new>
#include <numeric>

namespace fvx {

/* ---------------------------------------------------------------- kernel --------------- */

/// One row of a factor block as the registers hold it. pin() keeps the conversion to FP64 inside
/// the pass loop: hoisted out of it, the rows would take twice the registers.
template <class VT> struct FacRow;
template <> struct FacRow<double> {
	double2 a, b;
	__device__ __forceinline__ void load(const double* p)
	{
		a = reinterpret_cast<const double2*>(p)[0];
		b = reinterpret_cast<const double2*>(p)[1];
	}
	__device__ __forceinline__ void clear() { a = b = make_double2(0.0, 0.0); }
	__device__ __forceinline__ void get(double* v) const { v[0] = a.x; v[1] = a.y; v[2] = b.x; v[3] = b.y; }
	__device__ __forceinline__ void pin() {}
};
template <> struct FacRow<float> {
	float4 a;
	__device__ __forceinline__ void load(const float* p) { a = *reinterpret_cast<const float4*>(p); }
	__device__ __forceinline__ void clear() { a = make_float4(0, 0, 0, 0); }
	__device__ __forceinline__ void get(double* v) const { v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; }
	__device__ __forceinline__ void pin()
	{
		asm volatile("" : "+v"(a.x), "+v"(a.y), "+v"(a.z), "+v"(a.w));
	}
};
/// bfloat16 rows are widened to FP32 when they are loaded: unpacking in every pass costs 20
/// operations a cell.
template <> struct FacRow<bf16> : FacRow<float> {
	__device__ __forceinline__ void load(const bf16* p)
	{
		const uint2 w = *reinterpret_cast<const uint2*>(p);
		a = make_float4(__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
		                __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u));
	}
};

/// `npass` colour passes of workgroup p's patch; FIRST starts from zero instead of zin, its first
/// ncol passes reading lower colours only. A quad of lanes serves K of the patch's cells, lane q
/// holding row q of their five factor blocks in registers for the whole launch (NQ quads; FP64
/// K <= 2, else K <= 4: 126 registers at 1,024 threads), the iterates of patch and rim lie in
/// LDS, 32 bytes a cell, as do the right-hand sides and cell numbers.
///
/// rec[p][slot] = {cell (-1: none), bit e set: computed in the pass e passes before the last; bits
/// 26-29: the neighbour slots of lower colours; bit 30: the patch's own cell, LDS byte offsets of
/// the four neighbours' iterates}; an absent neighbour's is a zero (its factor block is zero
/// too). halo[p][h] = the cells only read (-1: none). Slots are in colour order, so that a wave
/// whose cells are all of another colour skips the pass.
///
/// Bound by the read of the factors of patch and rim (2.04 cells for one of the patch's own on 98,304
/// cells at three sweeps), beside which nothing runs: a workgroup fills its compute unit, loads its
/// rows, then makes the passes. A launch of three sweeps moves 55 MB with FP32 factors and takes
/// 16.9 us, 34 MB and 10.5 us with bfloat16, one of two sweeps 92 MB and 21 us with FP64: 10.6, 6.6
/// and 18 us of it at the rate of a large copy. The rest is the chain of passes (0.3 us each at
/// least: barrier, LDS and FMA latency; VALU issue 4 us, LDS 2 us in all) and the launch. 13 colour
/// passes take 58 us with FP32 factors. Sixteen instances read 503 MB of FP32 factors without any
/// rim, 98 us at that rate; a launch takes 111.
template <class VTF, int NQ, int K, bool FIRST>
__global__ __launch_bounds__(4*NQ)
void k_sgs_patch(int npass, int ncol, const uint4* __restrict__ rec,
                 const int* __restrict__ halo, int nhalo, const int* __restrict__ ilist, const VTF* __restrict__ fac, long sa,
                 const double* __restrict__ r, long sr, const double* __restrict__ zin, long szi,
                 double* __restrict__ zout, long szo)
{
	const long I = ilist ? ilist[blockIdx.y] : 0;
	if(I < 0) return;                     // a retired slot of a compacted list
	fac += I*sa; r += I*sr; zout += I*szo;
	if constexpr(!FIRST) zin += I*szi;
	extern __shared__ double zs[];
	double* rs = zs + 4*(K*NQ + 1 + nhalo);
	int* gs = reinterpret_cast<int*>(rs + 4*K*NQ);
	const int p = xcd_block();
	const int q = threadIdx.x & 3, j = threadIdx.x >> 2;
	rec += (size_t)p*K*NQ;
	FacRow<VTF> f[K][5];
	unsigned act[K], n01[K], n23[K];
#pragma unroll
	for(int k = 0; k < K; k++) {
		const uint4 c = rec[k*NQ + j];
		const int g = (int)c.x;
		act[k] = c.y; n01[k] = c.z; n23[k] = c.w;
#pragma unroll
		for(int s = 0; s < 5; s++) f[k][s].clear();
		double z0 = 0.0, r0 = 0.0;
		if(g >= 0) {
			const VTF* blk = fac + (size_t)g*80 + 4*q;
#pragma unroll
			for(int s = 0; s < 5; s++) f[k][s].load(blk + 16*s);
			r0 = r[4*g + q];
			if constexpr(!FIRST) z0 = zin[4*g + q];
		}
		zs[4*(k*NQ + j) + q] = z0;
		rs[4*(k*NQ + j) + q] = r0;
		if(q == 0) gs[k*NQ + j] = g;
	}
	for(int h = j; h < nhalo; h += NQ) {
		double z0 = 0.0;
		if constexpr(!FIRST) {
			const int g = halo[p*nhalo + h];
			if(g >= 0) z0 = zin[4*(long)g + q];
		}
		zs[4*(K*NQ + 1 + h) + q] = z0;
	}
	if(threadIdx.x < 4) zs[4*K*NQ + threadIdx.x] = 0.0;      // absent neighbours
	__syncthreads();
	const char* zb = reinterpret_cast<const char*>(zs);
	for(int e = npass - 1; e >= 0; e--) {
		const bool low = FIRST && e > npass - 1 - ncol;
#pragma unroll
		for(int k = 0; k < K; k++) {
			if((act[k] >> e) & 1u) {
				const unsigned off[4] = { n01[k] & 0xffffu, n01[k] >> 16, n23[k] & 0xffffu,
				                          n23[k] >> 16 };
				double t = rs[4*(k*NQ + j) + q], a[4], zv[4];
#pragma unroll
				for(int s = 0; s < 4; s++) {
					f[k][1 + s].pin();
					f[k][1 + s].get(a);
					load4(reinterpret_cast<const double*>(zb + off[s]), zv);
					double d = dot4(a, zv);
					if constexpr(FIRST) d = !low || ((act[k] >> (26 + s)) & 1u) ? d : 0.0;
					t -= d;
				}
				const double tv[4] = { quad_bcast<0>(t), quad_bcast<1>(t), quad_bcast<2>(t),
				                       quad_bcast<3>(t) };
				f[k][0].pin();
				f[k][0].get(a);
				zs[4*(k*NQ + j) + q] = dot4(a, tv);
			}
		}
		__syncthreads();
	}
#pragma unroll
	for(int k = 0; k < K; k++)
		if(act[k] >> 30) {
			const int g = gs[k*NQ + j];
			zout[4*(long)g + q] = zs[4*(k*NQ + j) + q];
		}
}

/* ---------------------------------------------------------------- patches -------------- */

namespace {

constexpr int SP_MAX_LOCAL = 2047;       // LDS byte offsets of 32-byte iterates in 16 bits
constexpr int SP_MAX_PASS = 26;          // pass bits of a record's second word
constexpr int SP_CUS = 256;              // compute units: one workgroup each

/// Computed cells a workgroup's registers hold: two (FP64) or four (FP32, and bfloat16 kept as
/// FP32) rows of five blocks per lane, 1,024 threads.
inline int capacity(int prec) { return prec == FVX_PREC_F64 ? 512 : 1024; }

inline int threads_for(int n) { return n < 1024 ? 1 : n < 8192 ? 4 : 8; }

/// The colour of the pass that is e passes before the last one of an application.
inline int pass_colour(int e, int ncol)
{
	const int per = 2*(ncol - 1), q = e % per;
	return q <= ncol - 1 ? q : per - q;
}

/// One patch: its own cells are cells_in[b, e); `cells` lists the computed ones by colour, within
/// a colour in the order they joined (the cells of late passes first), with their pass bits;
/// `halo` the cells only read.
struct Patch {
	std::vector<int> cells, halo;
	std::vector<unsigned> act;
	int b, e;
};

/// Divides the cells into compact patches and works out what each computes.
struct Patches {
	const fvx_pc_s& p;
	const int* nb;
	const int n, C, D, cap;
	std::vector<int> cells, da, db, set;
	std::vector<char> higher;              // the cell has a neighbour of a higher colour
	std::atomic<int> nset{1};
	struct Task { int b, e, id, np, from; };
	struct Work { std::vector<int> q, stamp, V; std::vector<unsigned> act; int mark = 0; };

	Patches(const fvx_pc_s& pc, const int* nbr, int cycles)
		: p(pc), nb(nbr), n(pc.m->nelem), C(pc.ncol), D(2*cycles*(C - 1) + 1), cap(capacity(pc.prec)),
		  cells(n), da(n), db(n), set(n, 0), higher(n, 0)
	{
		std::iota(cells.begin(), cells.end(), 0);
		for(int c = 0; c < n; c++)
			for(int k = 0; k < 4; k++) {
				const int o = nb[4*(size_t)c + k];
				if(o >= 0 && p.colour[o] > p.colour[c]) higher[c] = 1;
			}
	}

	/// Distances from `from` inside the task's cells, counted in cells (pieces not connected to
	/// it follow on); returns the cell reached last.
	int bfs(const Task& t, int from, std::vector<int>& d, std::vector<int>& q)
	{
		for(int i = t.b; i < t.e; i++) d[cells[i]] = -1;
		q.assign(1, from);
		d[from] = 0;
		size_t h = 0;
		for(int i = t.b;;) {
			for(; h < q.size(); h++) {
				const int c = q[h];
				for(int k = 0; k < 4; k++) {
					const int o = nb[4*(size_t)c + k];
					// other threads renumber the sets of their own cells only
					if(o >= 0 && __atomic_load_n(&set[o], __ATOMIC_RELAXED) == t.id && d[o] < 0) {
						d[o] = d[c] + 1;
						q.push_back(o);
					}
				}
			}
			if((int)q.size() == t.e - t.b) break;
			while(d[cells[i]] >= 0) i++;
			d[cells[i]] = d[q.back()] + 1;
			q.push_back(cells[i]);
		}
		return q.back();
	}

	/// Bisection across the longest direction, between an extreme cell of the division that made
	/// the set and the last cell a search from it reaches: the cells are divided by how much
	/// nearer they are to one end than to the other.
	void divide(const Task& t, std::vector<int>& q, Task& l, Task& r)
	{
		const int z = bfs(t, t.from, da, q);
		bfs(t, z, db, q);
		const int n1 = t.np/2, mid = t.b + (int)((long)(t.e - t.b)*n1/t.np);
		auto less = [&](int x, int y) {
			const int vx = da[x] - db[x], vy = da[y] - db[y];
			return vx != vy ? vx < vy : x < y;
		};
		std::nth_element(cells.begin() + t.b, cells.begin() + mid, cells.begin() + t.e, less);
		const int id = nset++;
		for(int i = mid; i < t.e; i++) __atomic_store_n(&set[cells[i]], id, __ATOMIC_RELAXED);
		l = Task{t.b, mid, t.id, n1, *std::min_element(cells.begin() + t.b, cells.begin() + mid, less)};
		r = Task{mid, t.e, id, t.np - n1,
		         *std::max_element(cells.begin() + mid, cells.begin() + t.e, less)};
	}

	/// What the patch of the task's cells computes in the D passes, from the last one back: the
	/// final values of its own cells need, in each pass, the cells of the pass's colour among
	/// those whose value is wanted after it, which adds their neighbours to the values wanted
	/// before it. On the way down the colours (0 < colour < the highest) only cells with a
	/// neighbour of a higher colour have changed neighbours since the way up.
	void grow(const Task& t, Work& w, Patch& x)
	{
		const int mark = ++w.mark;
		w.V.assign(cells.begin() + t.b, cells.begin() + t.e);
		for(int c : w.V) { w.stamp[c] = mark; w.act[c] = 0; }
		for(int e = 0; e < D; e++) {
			const int col = pass_colour(e, C), q = e % (2*(C - 1));
			const bool down = q > 0 && q < C - 1;
			const size_t cnt = w.V.size();
			for(size_t i = 0; i < cnt; i++) {
				const int c = w.V[i];
				if(p.colour[c] != col || (down && !higher[c])) continue;
				w.act[c] |= 1u << e;
				for(int k = 0; k < 4; k++) {
					const int o = nb[4*(size_t)c + k];
					if(o >= 0 && w.stamp[o] != mark) { w.stamp[o] = mark; w.act[o] = 0; w.V.push_back(o); }
				}
			}
		}
		x.b = t.b;
		x.e = t.e;
		for(int col = 0; col < C; col++)
			for(int c : w.V)
				if(w.act[c] && p.colour[c] == col) { x.cells.push_back(c); x.act.push_back(w.act[c]); }
		for(int c : w.V) if(!w.act[c]) x.halo.push_back(c);
	}

	/// About np patches of equal size; one that does not fit a workgroup is divided again.
	std::vector<Patch> run(int np)
	{
		std::vector<int> q;
		std::vector<Task> top(1, Task{0, n, 0, np, 0});
		top[0].from = bfs(top[0], 0, da, q);
		// the first divisions one after the other, the sets they give on threads of their own
		const int nt = threads_for(n);
		for(int k = 1; k < nt && np >= nt; k *= 2) {
			std::vector<Task> next(2*top.size());
			parallel((int)top.size(), [&](int i) {
				std::vector<int> qi;
				divide(top[i], qi, next[2*i], next[2*i + 1]);
			});
			top.swap(next);
		}
		std::vector<std::vector<Patch>> part(top.size());
		parallel((int)top.size(), [&](int i) {
			Work w;
			w.stamp.assign(n, 0);
			w.act.assign(n, 0);
			std::vector<Task> stack(1, top[i]);
			while(!stack.empty()) {
				Task t = stack.back(), l, r;
				stack.pop_back();
				if(t.np == 1) {
					Patch x;
					grow(t, w, x);
					if((int)x.cells.size() <= cap || t.e - t.b < 2) {
						part[i].push_back(std::move(x));
						continue;
					}
					t.np = 2;
				}
				divide(t, w.q, l, r);
				stack.push_back(r);
				stack.push_back(l);
			}
		});
		std::vector<Patch> out;
		for(auto& v : part) for(Patch& x : v) out.push_back(std::move(x));
		return out;
	}
};

struct Tables {
	std::vector<uint4> rec;
	std::vector<int> halo;
	int npatch = 0, slots = 0, nhalo = 0;
};

/// Records of about np patches for up to `cycles` sweeps per launch; false if one does not fit.
bool build(const fvx_pc_s& p, const std::vector<int>& nb, int np, int cycles, Tables& T)
{
	const int n = p.m->nelem;
	Patches P(p, nb.data(), cycles);
	const std::vector<Patch> pt = P.run(np);
	np = (int)pt.size();
	int most = 1;
	T.nhalo = 0;
	for(const Patch& x : pt) {
		most = std::max(most, (int)x.cells.size());
		T.nhalo = std::max(T.nhalo, (int)x.halo.size());
	}
	T.npatch = np;
	T.slots = most <= 128 ? 128 : (most + 255)/256*256;
	const int S = T.slots;
	if(most > P.cap || S + 1 + T.nhalo > SP_MAX_LOCAL) return false;
	T.rec.assign((size_t)np*S, make_uint4(0xffffffffu, 0, 0, 0));
	T.halo.assign(std::max((size_t)np*T.nhalo, (size_t)1), -1);
	const int nt = threads_for(n);
	parallel(nt, [&](int t) {
		std::vector<int> local(n);
		for(int b = (int)((long)np*t/nt); b < (int)((long)np*(t + 1)/nt); b++) {
			const Patch& x = pt[b];
			for(size_t i = 0; i < x.cells.size(); i++) local[x.cells[i]] = (int)i;
			for(size_t h = 0; h < x.halo.size(); h++) {
				local[x.halo[h]] = S + 1 + (int)h;
				T.halo[(size_t)b*T.nhalo + h] = x.halo[h];
			}
			for(size_t i = 0; i < x.cells.size(); i++) {
				const int c = x.cells[i];
				unsigned l[4], w = x.act[i];
				for(int k = 0; k < 4; k++) {
					const int o = nb[4*(size_t)c + k];
					l[k] = 32u*(unsigned)(o >= 0 ? local[o] : S);
					if(o >= 0 && p.colour[o] < p.colour[c]) w |= 1u << (SP_MAX_PASS + k);
				}
				T.rec[(size_t)b*S + i] = make_uint4((unsigned)c, w, l[0] | l[1] << 16,
				                                    l[2] | l[3] << 16);
			}
			for(int i = x.b; i < x.e; i++) T.rec[(size_t)b*S + local[P.cells[i]]].y |= 1u << 30;
		}
	});
	return true;
}

/// Computed cells of a patch of P cells, estimated: a compact set of cells grows by
/// 1.75 + 0.3 colours cells in diameter per sweep; most patches stay within 1.2 times the mean.
inline double computed(double P, int cycles, int ncol)
{
	const double d = std::sqrt(P) + (1.75 + 0.3*ncol)*cycles;
	return 1.2*d*d;
}

template <class VTF, int NQ, int K>
void launch(const fvx_pc_s& p, int npass, bool first, const VTF* fac, const double* r, long sr,
            const double* zin, long szi, double* zout, long szo, const Inst& L, hipStream_t s)
{
	const SgsPatch& t = p.patch;
	const size_t lds = 32*(size_t)(2*K*NQ + 1 + t.nhalo) + 4*(size_t)K*NQ;
	const dim3 g(t.npatch, L.nact);
	if(first)
		hipLaunchKernelGGL((k_sgs_patch<VTF, NQ, K, true>), g, dim3(4*NQ), lds, s, npass, p.ncol,
		                   t.d_rec.p, t.d_halo.p, t.nhalo, L.list, fac, 80L*p.m->nelem, r, sr,
		                   zin, szi, zout, szo);
	else
		hipLaunchKernelGGL((k_sgs_patch<VTF, NQ, K, false>), g, dim3(4*NQ), lds, s, npass, p.ncol,
		                   t.d_rec.p, t.d_halo.p, t.nhalo, L.list, fac, 80L*p.m->nelem, r, sr,
		                   zin, szi, zout, szo);
	FVX_HIP(hipGetLastError());
}

bool capturing(hipStream_t s)
{
	hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
	if(hipStreamIsCapturing(s, &st) != hipSuccess) { (void)hipGetLastError(); return true; }
	return st != hipStreamCaptureStatusNone;
}

/// Lets this thread allocate while another thread records a graph.
struct Relaxed {
	hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
	Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
	~Relaxed() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

template <class T> void upload(DBuf<T>& d, const std::vector<T>& h, hipStream_t s)
{
	d.alloc(h.size());
	FVX_HIP(hipMemcpyAsync(d.p, h.data(), h.size()*sizeof(T), hipMemcpyHostToDevice, s));
}

/* Which patches: the more sweeps a launch performs the fewer launches there are and the fewer
 * times the factors are read, but each sweep widens the rim of cells computed twice and uses up
 * the workgroup's registers. If every instance's patches fit the 256 compute units at once, the
 * largest number of sweeps (at most 4) whose patches fit; otherwise two sweeps on the largest
 * patches that fit. Per application (MI355X, colour passes -> patches): 48 cells FP64 x16 243 ->
 * 25 us; 4,608 cells 227 -> 37 us; 15,000 cells 234 -> 43 us; 98,304 cells FP64 360 -> 175, FP32
 * 294 -> 105, bfloat16 252 -> 86 us; 393,216 cells FP64 1,133 -> 644, FP32 848 -> 383 us;
 * 1,572,864 cells in Hilbert order (5 colours) FP64 6.63 -> 3.66, FP32 4.95 -> 2.15 ms. Other
 * choices measured on 98,304 cells: FP32 1 sweep per launch 165 us, 2 sweeps 112-119, 3 sweeps on
 * 414 smaller patches 133; FP64 1 sweep 304, 3 sweeps 214 us. A batch of 16 such instances (a few
 * pseudo-steps) FP32: 262 ms with colour passes; 186 / 142 / 148 with 1 / 2 / 3 sweeps. */
void make_tables(const fvx_pc_s& p, int most, hipStream_t s)
{
	SgsPatch& t = p.patch;
	const int C = p.ncol, n = p.m->nelem, cap = capacity(p.prec);
	t.cycles = 0;
	// 16 units are left for patches divided again
	double P = std::max(16.0, n/(double)std::max(1, (SP_CUS - 16)/p.ninst));
	int cycles = 0;
	for(int m = most; m >= std::min(2, most) && !cycles; m--)
		if(computed(P, m, C) <= cap) cycles = m;
	if(!cycles) {
		cycles = std::min(2, most);
		for(P = cap; P > 16 && computed(P, cycles, C) > cap;) P *= 0.95;
	}
	std::vector<int> nb(4*(size_t)n);
	for(int c = 0; c < n; c++)
		for(int k = 0; k < 4; k++) {
			const int o = k < p.m->nnode[c] ? p.m->esuel[4*(size_t)c + k] : -1;
			nb[4*(size_t)c + k] = o < n ? o : -1;
		}
	Tables T;
	if(!build(p, nb, std::max(1, (int)std::ceil(n/P)), cycles, T)) return;
	upload(t.d_rec, T.rec, s);
	upload(t.d_halo, T.halo, s);
	FVX_HIP(hipStreamSynchronize(s));
	t.slots = T.slots;
	t.npatch = T.npatch;
	t.nhalo = T.nhalo;
	t.cycles = cycles;
}

/// Sweeps per launch the tables should allow: at most 4, and their passes must fit a record's bits.
int most_sweeps(const fvx_pc_s& p)
{
	return std::min(std::min(4, p.sweeps), (SP_MAX_PASS - 1)/(2*(p.ncol - 1)));
}

/// Whether patches can serve the preconditioner on stream s at all.
bool possible(const fvx_pc_s& p, hipStream_t s)
{
	return p.type == FVX_PC_SGS && p.ncol > 1 && 2*(p.ncol - 1) + 1 <= SP_MAX_PASS && !p.patch.failed
	       && !capturing(s);
}

/// Runs f, which allocates; false where there is no memory: the colour passes then serve the handle.
template <class F> bool allocating(SgsPatch& t, F&& f)
{
	try {
		Relaxed relaxed;
		f();
		return true;
	}
	catch(const std::bad_alloc&) { t.failed = true; }
	catch(const Error& e) {
		t.failed = true;
		if(e.code != FVX_ERR_ALLOC) throw;
		(void)hipGetLastError();
	}
	return false;
}

void tables(const fvx_pc_s& p, int most, hipStream_t s)
{
	SgsPatch& t = p.patch;
	allocating(t, [&] {
		make_tables(p, most, s);
		t.most = most;
		t.spent = 0;
		if(!t.cycles) t.failed = true;
	});
}

/// Whether this application runs on the patches. The tables (made on the host: 2-4 ms for 4,608
/// cells, 8 ms for 98,304, 150-190 ms for 1,572,864) are made once the handle's applications have
/// taken about as long by colour passes as that takes, so that a preconditioner used a few times
/// does not pay for them; until then, and where the device has no memory for them, the colour passes
/// serve. The scratch vector of applications of more than one launch serves one stream between two
/// set-ups, and no recorded graph.
bool ready(const fvx_pc_s& p, size_t value, int nact, hipStream_t s)
{
	if(!possible(p, s)) return false;
	SgsPatch& t = p.patch;
	const int C = p.ncol, n = p.m->nelem, most = most_sweeps(p);
	if(t.most < most) {
		// us of a colour pass: a launch, and its share of the factors at ~7 TB/s
		t.spent += (2.0*p.sweeps*(C - 1) + 1)*(3.5 + 80.0*n*value*nact/C/7e6);
		if(t.spent >= 1500 + 0.07*n) tables(p, most, s);
	}
	if(t.failed || !t.cycles) return false;
	if(p.sweeps > t.cycles) {
		if(t.claimed && t.owner != s) return false;
		const size_t N = 4*(size_t)n*p.ninst;
		if(t.scratch.n != N && !allocating(t, [&] { t.scratch.alloc(N); })) return false;
		t.owner = s;
		t.claimed = true;
	}
	return true;
}

}

void sgs_patch_prepare(const fvx_pc_s& p, hipStream_t s)
{
	if(possible(p, s) && p.patch.most < most_sweeps(p)) tables(p, most_sweeps(p), s);
}

template <class VTF>
bool sgs_patch_apply(const fvx_pc_s& p, const VTF* fac, const double* r, long sr, double* z,
                     long sz, const Inst& L, hipStream_t s)
{
	SgsPatch& t = p.patch;
	if(r == z || !ready(p, sizeof(VTF), L.nact, s)) return false;
	const int steps = (p.sweeps + t.cycles - 1)/t.cycles;
	const long N = 4L*p.m->nelem;
	const double* zin = nullptr;
	long szi = 0;
	for(int i = 0, done = 0; i < steps; i++) {
		const int c = (p.sweeps - done + steps - i - 1)/(steps - i);
		done += c;
		const bool toz = (steps - 1 - i) % 2 == 0;
		double* zo = toz ? z : t.scratch.p;
		const long szo = toz ? sz : N;
		const int npass = 2*c*(p.ncol - 1) + (i == 0 ? 1 : 0);
#define FVX_SP(NQ, K) case NQ*K: \
			launch<VTF, NQ, K>(p, npass, i == 0, fac, r, sr, zin, szi, zo, szo, L, s); break;
		switch(t.slots) {
		FVX_SP(128, 1) FVX_SP(256, 1) FVX_SP(256, 2)
		default:
			if constexpr(sizeof(VTF) <= 4) switch(t.slots) {
			FVX_SP(256, 3) FVX_SP(256, 4)
			default: throw Error(FVX_ERR_INVALID, "no kernel for this patch size");
			}
			else throw Error(FVX_ERR_INVALID, "no kernel for this patch size");
		}
#undef FVX_SP
		zin = zo;
		szi = szo;
	}
	t.served++;
	return true;
}

template bool sgs_patch_apply<double>(const fvx_pc_s&, const double*, const double*, long, double*,
                                      long, const Inst&, hipStream_t);
template bool sgs_patch_apply<float>(const fvx_pc_s&, const float*, const double*, long, double*,
                                     long, const Inst&, hipStream_t);
template bool sgs_patch_apply<bf16>(const fvx_pc_s&, const bf16*, const double*, long, double*,
                                    long, const Inst&, hipStream_t);

}
