/* mpnn.hip -- learned warm start: a message-passing network over the cell graph that predicts
 * the converged state of an operating point, trained and evaluated by the kernels below.
 *
 * No reference counterpart: the reference starts a solve from the freestream or from a
 * first-order starter solve (src/utilities/casesolvers.cpp:225-386). The implicit solver still
 * decides the result: a predicted state is only an initial guess.
 *
 * Network (width 64, 4 layers; relu = max(0, .); bf16 weights, fp32 accumulation):
 *   h0 = x Wenc + benc                                  x: 8 node features
 *   P = hb Wa, Q = hb Wb                                hb: h rounded to bf16
 *   s_ik = P_i + Q_j + e_ik We + bm,  a_i = (1/deg_i) sum_k relu(s_ik)   (interior slots k)
 *   h' = h + relu(hb Wu + ab Wv + bu)                   ab: a rounded to bf16
 *   y = h4 Wdec + bdec                                  4 outputs per cell
 *
 * Data layout: rows are cells of G graphs (row = g*N + cell). Activations, Q, their gradients and
 * da are [rows][64] fp32 in the channel order of load_row; GEMM-only operands (a, dL/dpre,
 * dL/dP|dQ) bf16 in plain order. Per row and layer the relu patterns of the update (8 bytes) and
 * of the four messages (32 bytes) are kept for the backward pass.
 *
 * Matrix products run on the MFMA units (v_mfma_f32_16x16x32_bf16), one 16-row tile per wavefront
 * at a time with the weights' B fragments in LDS; a launch is a whole layer, forward or backward.
 * Weight gradients (A^T B over all rows) stage 64-row chunks transposed in LDS and write one
 * partial per workgroup; partials are summed in a fixed order, so every result is deterministic.
 */
#include "fvx_internal.hpp"
#include "wave.hpp"
#include <algorithm>
#include <cmath>

namespace fvx {
namespace mpnn {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16_t;

constexpr int RB = 256;                 // threads per workgroup of every kernel here
constexpr int TILE_BLOCKS = 768;        // workgroup cap of the row-tile kernels
constexpr int RED_BLOCKS = 512;         // workgroups that write reduction partials

__device__ __forceinline__ bf16_t f2bf(float f)
{
	unsigned u = __float_as_uint(f);
	u += 0x7FFFu + ((u >> 16) & 1u);
	return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t b) { return __uint_as_float((unsigned)b << 16); }
__device__ __forceinline__ unsigned pack2(float a, float b)
{
	return (unsigned)f2bf(a) | ((unsigned)f2bf(b) << 16);
}
__device__ __forceinline__ bf16x8 to_frag(const float* v)
{
	const u32x4 u = { pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]) };
	return __builtin_bit_cast(bf16x8, u);
}
__device__ __forceinline__ void load8(const float* p, float* v)
{
	const f32x4 a = *reinterpret_cast<const f32x4*>(p);
	const f32x4 b = *reinterpret_cast<const f32x4*>(p + 4);
	v[0] = a[0]; v[1] = a[1]; v[2] = a[2]; v[3] = a[3];
	v[4] = b[0]; v[5] = b[1]; v[6] = b[2]; v[7] = b[3];
}
__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c)
{
	return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

/// Arguments shared by the kernels of one pass.
struct Graph {
	int N;                  // cells per graph
	int R;                  // rows = graphs x N
	const int* nbr;         // [N][4] interior neighbour or -1
	const int* rev;         // [N][4] slot of this cell in the neighbour's list
	const float* invdeg;    // [N]
	const float* stat;      // [N][6] static node features
	const float* edge;      // [N][4][4] edge features
	const float* gfeat;     // [G][2] per-graph features
};

// ------------------------------------------------------------------------------------------
// weight packing: fp32 master -> bf16-rounded copy (VALU weights) and MFMA B fragments
// ------------------------------------------------------------------------------------------

/// B-operand element (k, n) of packed matrix `mat` of layer l (see the file header).
__device__ __forceinline__ float bmat(const float* w, int l, int mat, int k, int n)
{
	const float* L = w + OFF_L0 + l*LSZ;
	switch(mat) {
	case M_PQ:   return n < W ? L[L_WA + k*W + n] : L[L_WB + k*W + n - W];
	case M_UPD:  return k < W ? L[L_WU + k*W + n] : L[L_WV + (k - W)*W + n];
	case M_BUPD: return n < W ? L[L_WU + n*W + k] : L[L_WV + (n - W)*W + k];
	default:     return k < W ? L[L_WA + n*W + k] : L[L_WB + n*W + k - W];
	}
}

__global__ void __launch_bounds__(RB) k_pack(const float* __restrict__ w, float* __restrict__ wq,
                                             bf16_t* __restrict__ frag)
{
	const int t = blockIdx.x*RB + threadIdx.x;
	if(t < NPARAM) {
		// matrices enter the arithmetic rounded to bf16, biases unchanged
		const bool bias = (t >= OFF_BENC && t < OFF_L0) || t >= OFF_BDEC
		                  || (t >= OFF_L0 && t < OFF_WDEC
		                      && (((t - OFF_L0) % LSZ >= L_BM && (t - OFF_L0) % LSZ < L_WU)
		                          || (t - OFF_L0) % LSZ >= L_BU));
		wq[t] = bias ? w[t] : bf2f(f2bf(w[t]));
	}
	if(t < NL*4*FRAG_MAT) {
		const int lm = t / FRAG_MAT, r = t % FRAG_MAT;
		const int l = lm / 4, mat = lm % 4;
		const int e = r % 8, lane = (r / 8) % 64, sj = r / 512;
		const int nt = (mat == M_PQ || mat == M_BUPD) ? 8 : 4;
		const int s = sj / nt, j = sj % nt;
		const int k = 32*s + 8*(lane/16) + e, n = 16*j + lane%16;
		frag[t] = f2bf(bmat(w, l, mat, k, n));
	}
}

// ------------------------------------------------------------------------------------------
// row tiles: a wavefront takes 16 rows at a time. A operands (and everything loaded from or
// stored to row-major arrays) are in the A layout -- lane holds row lane & 15, channels
// 32 s + 8 (lane >> 4) .. + 7 of slice s --, products come in the C layout -- rows
// 4 (lane >> 4) + q, channel 16 j + (lane & 15). A 16 x 64 tile in LDS, private to the wave, turns
// one into the other. The weight fragments lie in LDS for all waves of the workgroup: in
// registers (64-128 of them) they left two waves per SIMD.
// ------------------------------------------------------------------------------------------

constexpr int TLD = 68;                 // floats per tile row: both layouts free of bank conflicts
constexpr int TILE = 16*TLD;
constexpr int WAVES = RB/64;

/// Scalar: a branch on it must not leave an MFMA to the exec mask, which it ignores.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
__device__ __forceinline__ void wave_sync()
{
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
}
__device__ __forceinline__ void tile_put_c(float* t, int lane, const f32x4* acc)
{
	wave_sync();
#pragma unroll
	for(int j = 0; j < 4; j++)
#pragma unroll
		for(int q = 0; q < 4; q++) t[(4*(lane >> 4) + q)*TLD + 16*j + (lane & 15)] = acc[j][q];
	wave_sync();
}
__device__ __forceinline__ void tile_get_a(const float* t, int lane, int s, float* v)
{
	load8(t + (lane & 15)*TLD + 32*s + 8*(lane >> 4), v);
}
/// fp32 rows (h, Q, da, the gradients) are kept in an order of their own: position 32 s + 16 b +
/// 4 g + i holds channel 32 s + 8 g + 4 b + i, so that each of the two 16-byte accesses of a lane's
/// 8 channels makes, with the other lane groups, a full 64-byte segment of every row. In channel
/// order every access touched twice the segments: k_layer_bwd took 643 us instead of 565 (at two
/// waves per SIMD).
__device__ __forceinline__ void load_row(const float* __restrict__ rows, size_t r, int s, int lane,
                                         float* v)
{
	const float* p = rows + r*W + 32*s + 4*(lane >> 4);
	const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 16);
#pragma unroll
	for(int e = 0; e < 4; e++) { v[e] = a[e]; v[4 + e] = b[e]; }
}
__device__ __forceinline__ void store_row(float* __restrict__ rows, size_t r, int s, int lane,
                                          const float* v)
{
	float* p = rows + r*W + 32*s + 4*(lane >> 4);
	*reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
	*reinterpret_cast<f32x4*>(p + 16) = f32x4{v[4], v[5], v[6], v[7]};
}
/// Channel at position p of a row.
__device__ __forceinline__ int chan(int p) { return (p & 35) | ((p & 12) << 1) | ((p & 16) >> 2); }

/// acc[j] = sum over S slices of a[s] x the fragments f[(s*NT + J0 + j)*64 ..] in LDS, j < 4.
template <int S, int NT, int J0 = 0>
__device__ __forceinline__ void tile_mm(const bf16x8* f, int lane, const bf16x8* a, f32x4* acc)
{
#pragma unroll
	for(int j = 0; j < 4; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
	for(int s = 0; s < S; s++)
#pragma unroll
		for(int j = 0; j < 4; j++) acc[j] = mfma(a[s], f[(s*NT + J0 + j)*64 + lane], acc[j]);
}

template <int CTRL> __device__ __forceinline__ float dpp_f(float v)
{
	return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xF,
	                                                          0xF, false));
}
/// Sum of v[e] over the 16 rows (lanes of equal lane >> 4), for e = lane & 7. Halves the values in
/// each exchange: 29 instructions for 8 sums, and one register per sum to keep them over the tiles.
__device__ __forceinline__ float row_sums8(int lane, const float (&v)[8])
{
	const bool h4 = lane & 4, h2 = lane & 2, h1 = lane & 1;
	float a[8], b[4], c[2];
#pragma unroll
	for(int e = 0; e < 8; e++) a[e] = v[e] + dpp_f<0x128>(v[e]);              // row_ror:8
#pragma unroll
	for(int e = 0; e < 4; e++)
		b[e] = (h4 ? a[4 + e] : a[e]) + dpp_f<0x141>(h4 ? a[e] : a[4 + e]);    // row_half_mirror
#pragma unroll
	for(int e = 0; e < 2; e++)
		c[e] = (h2 ? b[2 + e] : b[e]) + dpp_f<0x4E>(h2 ? b[e] : b[2 + e]);     // lane ^ 2
	return (h1 ? c[1] : c[0]) + dpp_f<0xB1>(h1 ? c[0] : c[1]);               // lane ^ 1
}

/// Fragments [s][j0 .. j0 + nj) of a packed matrix of NT columns of fragments to LDS.
__device__ __forceinline__ void stage_frags(bf16x8* dst, const bf16_t* __restrict__ frag, int S,
                                            int NT, int j0, int nj)
{
	const bf16x8* src = reinterpret_cast<const bf16x8*>(frag);
	for(int i = threadIdx.x; i < S*nj*64; i += RB) {
		const int l = i & 63, f = i >> 6, s = f/nj, j = f - s*nj;
		dst[i] = src[(s*NT + j0 + j)*64 + l];
	}
}

/// The tiles of a wavefront: every XCD owns a contiguous range and its wavefronts walk it side by
/// side, so that the rows gathered from neighbouring cells are mostly in its L2 (a contiguous range
/// per workgroup: k_layer 299 us instead of 274 on 786,432 rows).
struct Tiles { int t, end, step; };
__device__ __forceinline__ Tiles my_tiles(int ntile)
{
	const int nb = gridDim.x, nx = min(nb, 8), x = blockIdx.x % nx, local = blockIdx.x/nx;
	const int wgs = nb/nx + (x < nb % nx), per = (ntile + nx - 1)/nx;
	const int wave = wave_id();
	return { x*per + local*WAVES + wave, min((x + 1)*per, ntile), wgs*WAVES };
}

__device__ __forceinline__ void node_x(const Graph& g, int r, float* x)
{
	const int node = r % g.N, gi = r / g.N;
#pragma unroll
	for(int f = 0; f < NSTAT; f++) x[f] = g.stat[node*NSTAT + f];
	x[6] = g.gfeat[2*gi];
	x[7] = g.gfeat[2*gi + 1];
}

/// h0 = x Wenc + benc and Q0 = h0b Wb of the first layer.
__global__ void __launch_bounds__(RB) k_embed(Graph g, int ntile, const float* __restrict__ wq,
                                              const bf16_t* __restrict__ fpq,
                                              float* __restrict__ h0, float* __restrict__ q0)
{
	__shared__ bf16x8 wf[8*64];
	__shared__ __attribute__((aligned(16))) float we[(FIN + 1)*W], tile[WAVES*TILE];
	stage_frags(wf, fpq, 2, 8, 4, 4);
	for(int i = threadIdx.x; i < (FIN + 1)*W; i += RB)
		we[i] = i < FIN*W ? wq[OFF_WENC + i] : wq[OFF_BENC + i - FIN*W];
	__syncthreads();
	const int lane = threadIdx.x & 63, wave = wave_id();
	float* t = tile + wave*TILE;
	const Tiles ts = my_tiles(ntile);
	for(int tt = ts.t; tt < ts.end; tt += ts.step) {
		const int r = 16*tt + (lane & 15), rc = min(r, g.R - 1);
		float x[FIN];
		node_x(g, rc, x);
		bf16x8 a[2];
#pragma unroll
		for(int s = 0; s < 2; s++) {
			const int c0 = 32*s + 8*(lane >> 4);
			float v[8], w[8];
			load8(we + FIN*W + c0, v);
#pragma unroll
			for(int f = 0; f < FIN; f++) {
				load8(we + f*W + c0, w);
#pragma unroll
				for(int e = 0; e < 8; e++) v[e] += x[f]*w[e];
			}
			if(r < g.R) store_row(h0, r, s, lane, v);
			a[s] = to_frag(v);
		}
		f32x4 acc[4];
		tile_mm<2, 4>(wf, lane, a, acc);
		tile_put_c(t, lane, acc);
#pragma unroll
		for(int s = 0; s < 2; s++) {
			float v[8];
			tile_get_a(t, lane, s, v);
			if(r < g.R) store_row(q0, r, s, lane, v);
		}
	}
}

/// Backward of the update, from the gradient gn of its output rows and its relu mask (A layout,
/// both slices; mk[s] bit e): dpre = gn * mask (kept as bf16), [dh_part | da] = dpre [Wu^T | Wv^T],
/// gpart = gn + dh_part, and da is multiplied by the 1/deg (id) of the mean.
__device__ __forceinline__ void update_bwd_tile(const bf16x8* wf, float* t, int lane, int r, bool ok,
                                                const float (&gn)[2][8], const unsigned (&mk)[2],
                                                float id, bf16_t* __restrict__ dpre,
                                                float* __restrict__ gpart, float* __restrict__ da)
{
	bf16x8 a[2];
#pragma unroll
	for(int s = 0; s < 2; s++) {
		float v[8];
#pragma unroll
		for(int e = 0; e < 8; e++) v[e] = (mk[s] >> e) & 1u ? gn[s][e] : 0.f;
		a[s] = to_frag(v);
		if(ok) *reinterpret_cast<bf16x8*>(dpre + (size_t)r*W + 32*s + 8*(lane >> 4)) = a[s];
	}
	f32x4 acc[4];
	tile_mm<2, 8>(wf, lane, a, acc);
	tile_put_c(t, lane, acc);
#pragma unroll
	for(int s = 0; s < 2; s++) {
		float v[8];
		tile_get_a(t, lane, s, v);
#pragma unroll
		for(int e = 0; e < 8; e++) v[e] = gn[s][e] + v[e];
		if(ok) store_row(gpart, r, s, lane, v);
	}
	tile_mm<2, 8, 4>(wf, lane, a, acc);
	tile_put_c(t, lane, acc);
#pragma unroll
	for(int s = 0; s < 2; s++) {
		float v[8];
		tile_get_a(t, lane, s, v);
#pragma unroll
		for(int e = 0; e < 8; e++) v[e] *= id;
		if(ok) store_row(da, r, s, lane, v);
	}
}

/// One layer: P = hb Wa (kept in the wave), messages and their mean a over the cell's slots from
/// the neighbours' Q, h_out = h + relu([hb | ab] [Wu; Wv] + bu), and the next layer's
/// Q = h_outb Wb. TRAIN keeps ab, the relu mask of the update (byte [row][s][lane >> 4]) and those
/// of the messages (word [row][s][lane >> 4], byte k = slot k).
/// LAST goes on with the decoder y = h_out Wdec + bdec instead of storing h_out and Q. In inference
/// y is the result. In training the targets of graph gi are rows ids[gi] of the target set and
/// dy = 2 (y - t) inv_count, gn = dy Wdec^T goes through the backward of the update (update_bwd_tile)
/// right here, and workgroup partials of dWdec, dbdec and the squared error are left in part.
///
/// Bound by HBM and the gathers: per row h 256 + Q about 256 + edges 80 read, h 256 + Q 256
/// (+ 168 in training) written. P|Q written by a launch of its own and read back took 565 us per
/// layer on 786,432 rows (117 + 449), this takes 277 (1.1 GB, 77% of the copy rate). Three workgroups a
/// compute unit (168 registers; in inference 52 bytes a lane spill, 56 in LAST), two (by LDS) for LAST
/// in training, which takes 345 us with the decoder and its backward pass (in launches of their own
/// 620: 277 + 198 + 152). One graph of 98,304 cells, 34 us a layer: two tiles a wave, too few to hide
/// the gathers.
template <bool TRAIN, bool LAST>
__global__ void __launch_bounds__(RB, TRAIN && LAST ? 2 : 3)
k_layer(Graph g, int ntile, const float* __restrict__ h, const float* __restrict__ q,
        const float* __restrict__ wl, const bf16_t* __restrict__ fpq, const bf16_t* __restrict__ fupd,
        const bf16_t* __restrict__ fnext, const float* __restrict__ wq,
        float* __restrict__ hout, float* __restrict__ qout,                       // !LAST
        bf16_t* __restrict__ ab, unsigned char* __restrict__ umask, unsigned* __restrict__ mmask, // TRAIN
        float* __restrict__ y,                                                    // LAST, inference
        const float* __restrict__ tgt, const int* __restrict__ ids, double inv_count, // LAST, training
        bf16_t* __restrict__ dpre, float* __restrict__ gpart, float* __restrict__ da,
        float* __restrict__ part)
{
	constexpr int NF = !LAST ? 32 : TRAIN ? 40 : 24;
	__shared__ bf16x8 wf[NF*64];
	__shared__ __attribute__((aligned(16))) float we[6*W], tile[WAVES*TILE];
	__shared__ __attribute__((aligned(16))) float wd[LAST ? FO*W + FO : 1];
	stage_frags(wf, fpq, 2, 8, 0, 4);
	stage_frags(wf + 8*64, fupd, 4, 4, 0, 4);
	if constexpr(!LAST) stage_frags(wf + 24*64, fnext, 2, 8, 4, 4);      // the next layer's Wb
	else if constexpr(TRAIN) stage_frags(wf + 24*64, fnext, 2, 8, 0, 8); // this layer's [Wu^T|Wv^T]
	for(int i = threadIdx.x; i < 6*W; i += RB)      // We, bm, bu
		we[i] = wl[i < 4*W ? L_WE + i : i < 5*W ? L_BM + i - 4*W : L_BU + i - 5*W];
	if constexpr(LAST)
		for(int i = threadIdx.x; i < FO*W + FO; i += RB) wd[i] = wq[OFF_WDEC + i];
	__syncthreads();
	const int lane = threadIdx.x & 63, wave = wave_id(), R = g.R;
	float* t = tile + wave*TILE;
	float dsum[2][FO] = {}, dacc[5] = {0.f, 0.f, 0.f, 0.f, 0.f};
	const Tiles ts = my_tiles(ntile);
	for(int tt = ts.t; tt < ts.end; tt += ts.step) {
		const int r = 16*tt + (lane & 15), rc = min(r, R - 1);
		const int node = rc % g.N;
		const size_t base = (size_t)(rc - node);
		float hv[2][8];
		bf16x8 a[4];
#pragma unroll
		for(int s = 0; s < 2; s++) {
			load_row(h, rc, s, lane, hv[s]);
			a[s] = to_frag(hv[s]);
		}
		const int4 nb = *reinterpret_cast<const int4*>(g.nbr + 4*node);
		const int nbs[4] = { nb.x, nb.y, nb.z, nb.w };
		f32x4 ef[4];
#pragma unroll
		for(int k = 0; k < 4; k++)
			ef[k] = *reinterpret_cast<const f32x4*>(g.edge + ((size_t)node*4 + k)*4);
		const float id = g.invdeg[node];
		f32x4 acc[4];
		tile_mm<2, 4>(wf, lane, a, acc);
		tile_put_c(t, lane, acc);
		unsigned mm[2] = {0u, 0u};
#pragma unroll
		for(int s = 0; s < 2; s++) {
			const int c0 = 32*s + 8*(lane >> 4);
			float p[8], qv[4][8], w[4][8], bm[8], av[8];
#pragma unroll
			for(int k = 0; k < 4; k++)
				load_row(q, base + (nbs[k] >= 0 ? nbs[k] : node), s, lane, qv[k]);
			tile_get_a(t, lane, s, p);
#pragma unroll
			for(int f = 0; f < 4; f++) load8(we + f*W + c0, w[f]);
			load8(we + 4*W + c0, bm);
#pragma unroll
			for(int e = 0; e < 8; e++) av[e] = 0.f;
#pragma unroll
			for(int k = 0; k < 4; k++) {
				const bool on = nbs[k] >= 0;
				unsigned bits = 0u;
#pragma unroll
				for(int e = 0; e < 8; e++) {
					const float m = p[e] + qv[k][e] + (ef[k][0]*w[0][e] + ef[k][1]*w[1][e]
					                                   + ef[k][2]*w[2][e] + ef[k][3]*w[3][e]) + bm[e];
					av[e] += on ? fmaxf(m, 0.f) : 0.f;
					if constexpr(TRAIN) bits |= m > 0.f ? 1u << e : 0u;
				}
				if constexpr(TRAIN) mm[s] |= on ? bits << 8*k : 0u;
			}
#pragma unroll
			for(int e = 0; e < 8; e++) av[e] *= id;
			a[2 + s] = to_frag(av);
			if constexpr(TRAIN) {
				if(r < R) {
					*reinterpret_cast<bf16x8*>(ab + (size_t)r*W + c0) = a[2 + s];
					mmask[(size_t)r*8 + 4*s + (lane >> 4)] = mm[s];
				}
			}
		}
		tile_mm<4, 4>(wf + 8*64, lane, a, acc);
#pragma unroll
		for(int j = 0; j < 4; j++) {
			const float bu = we[5*W + 16*j + (lane & 15)];
#pragma unroll
			for(int i = 0; i < 4; i++) acc[j][i] = fmaxf(acc[j][i] + bu, 0.f);
		}
		tile_put_c(t, lane, acc);
		float yo[FO] = {0.f, 0.f, 0.f, 0.f};
		unsigned um[2];
#pragma unroll
		for(int s = 0; s < 2; s++) {
			const int c0 = 32*s + 8*(lane >> 4);
			float u[8];
			tile_get_a(t, lane, s, u);
			um[s] = 0u;
#pragma unroll
			for(int e = 0; e < 8; e++) {
				if constexpr(TRAIN) um[s] |= u[e] > 0.f ? 1u << e : 0u;
				hv[s][e] = hv[s][e] + u[e];
			}
			if constexpr(!LAST) {
				if(r < R) store_row(hout, r, s, lane, hv[s]);
				if(TRAIN && r < R) umask[(size_t)r*8 + 4*s + (lane >> 4)] = (unsigned char)um[s];
				a[s] = to_frag(hv[s]);
			} else {
#pragma unroll
				for(int e = 0; e < 8; e++) {
					const f32x4 d = *reinterpret_cast<const f32x4*>(wd + (c0 + e)*FO);
#pragma unroll
					for(int o = 0; o < FO; o++) yo[o] += hv[s][e]*d[o];
				}
			}
		}
		if constexpr(!LAST) {
			tile_mm<2, 4>(wf + 24*64, lane, a, acc);
			tile_put_c(t, lane, acc);
#pragma unroll
			for(int s = 0; s < 2; s++) {
				float v[8];
				tile_get_a(t, lane, s, v);
				if(r < R) store_row(qout, r, s, lane, v);
			}
		} else {
#pragma unroll
			for(int o = 0; o < FO; o++) {
				yo[o] += __shfl_xor(yo[o], 16);
				yo[o] += __shfl_xor(yo[o], 32);
				yo[o] += wd[FO*W + o];
			}
			if constexpr(!TRAIN) {
				if(lane < 16 && r < R)
					*reinterpret_cast<f32x4*>(y + (size_t)r*FO) = f32x4{yo[0], yo[1], yo[2], yo[3]};
			} else {
				const f32x4 tv = *reinterpret_cast<const f32x4*>(tgt + ((size_t)ids[rc/g.N]*g.N + node)*FO);
				float dy[FO], gn[2][8];
#pragma unroll
				for(int o = 0; o < FO; o++) {
					const float d = r < R ? yo[o] - tv[o] : 0.f;
					dy[o] = (float)(2.0*(double)d*inv_count);
					dacc[o] += dy[o];
					dacc[4] += d*d;
				}
#pragma unroll
				for(int s = 0; s < 2; s++)
#pragma unroll
					for(int e = 0; e < 8; e++) {
						const f32x4 d = *reinterpret_cast<const f32x4*>(wd + (32*s + 8*(lane >> 4) + e)*FO);
						gn[s][e] = dy[0]*d[0] + dy[1]*d[1] + dy[2]*d[2] + dy[3]*d[3];
					}
#pragma unroll
				for(int s = 0; s < 2; s++)
#pragma unroll
					for(int o = 0; o < FO; o++) {
						float v[8];
#pragma unroll
						for(int e = 0; e < 8; e++) v[e] = hv[s][e]*dy[o];
						dsum[s][o] += row_sums8(lane, v);
					}
				update_bwd_tile(wf + 24*64, t, lane, r, r < R, gn, um, id, dpre, gpart, da);
			}
		}
	}
	if constexpr(TRAIN && LAST) {
		// partial layout: Wdec[c][o] (256), bdec (4), squared error (1)
		float* red = t;
		wave_sync();
#pragma unroll
		for(int s = 0; s < 2; s++)
#pragma unroll
			for(int o = 0; o < FO; o++)
				if((lane & 15) < 8) red[(32*s + 8*(lane >> 4) + (lane & 7))*FO + o] = dsum[s][o];
#pragma unroll
		for(int i = 0; i < 5; i++) {
			float v = dacc[i];
			v += __shfl_xor(v, 8);
			v += __shfl_xor(v, 4);
			v += __shfl_xor(v, 2);
			v += __shfl_xor(v, 1);
			if(lane == 0) red[256 + i] = v;
		}
		__syncthreads();
		for(int i = threadIdx.x; i < 261; i += RB) {
			float v = 0.f;
			for(int w = 0; w < WAVES; w++) v += tile[w*TILE + i];
			part[(size_t)blockIdx.x*261 + i] = v;
		}
	}
}

/// Backward through one layer's messages and P|Q, and through the previous layer's update.
///   ds_ik = da_i [s_ik > 0] (the forward pass's masks; da holds the factor 1/deg already);
///   dP_i = sum_k ds_ik;
///   dQ_i = sum over the slots of i of ds at the neighbour's reverse slot;
///   gn = gpart + [dP | dQ] [Wa^T; Wb^T], the gradient of the layer's input;
/// then update_bwd_tile with the previous layer's mask and weights (FIRST: gn itself is written,
/// for the encoder). dP|dQ are kept as bf16 (an operand of the weight gradients); workgroup
/// partials of dWe = sum e_ik ds_ik and dbm = sum dP.
///
/// Bound by HBM and the gathers of da: per row da 256 + about 256 + masks 64 + edges 80 + gpart 256
/// read, dP|dQ 256 + dpre 128 + gpart 256 + da 256 written. Three launches that recomputed the
/// messages from P|Q took 1,148 us per layer on 786,432 rows (790 + 166 + 192), this takes 403
/// (1.5 GB, 71% of the copy rate). Three waves per SIMD, with 36 bytes a lane of spills (none in
/// FIRST): with the sums of dWe and dbm kept per lane and row (80 registers) instead of added over the
/// rows of each tile, two waves took 565.
template <bool FIRST>
__global__ void __launch_bounds__(RB, 3) k_layer_bwd(Graph g, int ntile,
                                                     const float* __restrict__ da,
                                                     const unsigned* __restrict__ mmask,
                                                     const bf16_t* __restrict__ fbpq,
                                                     const bf16_t* __restrict__ fbupd,
                                                     const unsigned char* __restrict__ umask,
                                                     bf16_t* __restrict__ dpq,
                                                     float* __restrict__ gpart,
                                                     bf16_t* __restrict__ dpre,
                                                     float* __restrict__ daout,
                                                     float* __restrict__ part)
{
	__shared__ bf16x8 wf[(FIRST ? 16 : 32)*64];
	__shared__ __attribute__((aligned(16))) float tile[WAVES*TILE];
	stage_frags(wf, fbpq, 4, 4, 0, 4);
	if constexpr(!FIRST) stage_frags(wf + 16*64, fbupd, 2, 8, 0, 8);
	__syncthreads();
	const int lane = threadIdx.x & 63, wave = wave_id(), R = g.R, gl = lane >> 4;
	float* t = tile + wave*TILE;
	float wsum[5][2];
#pragma unroll
	for(int f = 0; f < 5; f++) wsum[f][0] = wsum[f][1] = 0.f;
	const Tiles ts = my_tiles(ntile);
	for(int tt = ts.t; tt < ts.end; tt += ts.step) {
		const int r = 16*tt + (lane & 15), rc = min(r, R - 1);
		const bool ok = r < R;
		const int node = rc % g.N;
		const size_t base = (size_t)(rc - node);
		const int4 nb = *reinterpret_cast<const int4*>(g.nbr + 4*node);
		const int4 rv = *reinterpret_cast<const int4*>(g.rev + 4*node);
		const int nbs[4] = { nb.x, nb.y, nb.z, nb.w }, rvs[4] = { rv.x, rv.y, rv.z, rv.w };
		size_t rj[4];
#pragma unroll
		for(int k = 0; k < 4; k++) {
			rj[k] = base + (nbs[k] >= 0 ? nbs[k] : node);
		}
		bf16x8 a[4];
#pragma unroll
		for(int s = 0; s < 2; s++) {
			const int c0 = 32*s + 8*gl;
			float d[8], dn[4][8], dP[8], dQ[8];
			load_row(da, rc, s, lane, d);
			// a row past the end contributes nothing
			const unsigned mo = ok ? mmask[(size_t)rc*8 + 4*s + gl] : 0u;
			unsigned mn[4];
#pragma unroll
			for(int k = 0; k < 4; k++) {
				load_row(da, rj[k], s, lane, dn[k]);
				mn[k] = mmask[rj[k]*8 + 4*s + gl] >> 8*(rvs[k] & 3);
				if(nbs[k] < 0) mn[k] = 0u;
			}
#pragma unroll
			for(int e = 0; e < 8; e++) { dP[e] = 0.f; dQ[e] = 0.f; }
			float we[4][8];
#pragma unroll
			for(int f = 0; f < 4; f++)
#pragma unroll
				for(int e = 0; e < 8; e++) we[f][e] = 0.f;
#pragma unroll
			for(int k = 0; k < 4; k++) {
				const f32x4 ef = *reinterpret_cast<const f32x4*>(g.edge + ((size_t)node*4 + k)*4);
#pragma unroll
				for(int e = 0; e < 8; e++) {
					const float ds = (mo >> (8*k + e)) & 1u ? d[e] : 0.f;
					dP[e] += ds;
#pragma unroll
					for(int f = 0; f < 4; f++) we[f][e] += ef[f]*ds;
					dQ[e] += (mn[k] >> e) & 1u ? dn[k][e] : 0.f;
				}
			}
#pragma unroll
			for(int f = 0; f < 4; f++) wsum[f][s] += row_sums8(lane, we[f]);
			wsum[4][s] += row_sums8(lane, dP);
			a[s] = to_frag(dP);
			a[2 + s] = to_frag(dQ);
			if(ok) {
				*reinterpret_cast<bf16x8*>(dpq + (size_t)r*2*W + c0) = a[s];
				*reinterpret_cast<bf16x8*>(dpq + (size_t)r*2*W + W + c0) = a[2 + s];
			}
		}
		f32x4 acc[4];
		tile_mm<4, 4>(wf, lane, a, acc);
		tile_put_c(t, lane, acc);
		float gn[2][8];
#pragma unroll
		for(int s = 0; s < 2; s++) {
			float v[8];
			tile_get_a(t, lane, s, v);
			load_row(gpart, rc, s, lane, gn[s]);
#pragma unroll
			for(int e = 0; e < 8; e++) gn[s][e] = gn[s][e] + v[e];
			if constexpr(FIRST) { if(ok) store_row(gpart, r, s, lane, gn[s]); }
		}
		if constexpr(!FIRST) {
			const unsigned mk[2] = { umask[(size_t)rc*8 + gl], umask[(size_t)rc*8 + 4 + gl] };
			update_bwd_tile(wf + 16*64, t, lane, r, ok, gn, mk, g.invdeg[node], dpre, gpart, daout);
		}
	}
	// partial layout: We[f][c] (256), bm[c] (64), added over the waves in order
	wave_sync();
#pragma unroll
	for(int f = 0; f < 5; f++)
#pragma unroll
		for(int s = 0; s < 2; s++)
			if((lane & 15) < 8) t[f*W + 32*s + 8*gl + (lane & 7)] = wsum[f][s];
	__syncthreads();
	for(int i = threadIdx.x; i < 320; i += RB) {
		float s = 0.f;
		for(int w = 0; w < WAVES; w++) s += tile[w*TILE + i];
		part[(size_t)blockIdx.x*320 + i] = s;
	}
}

/// Encoder backward partials: dWenc[f][c] = sum_r x_f g0[r][c], dbenc[c] = sum_r g0[r][c];
/// 16 lanes per row, 4 channels each. Bound by the read of g0: one row per wave at a time took
/// 284 us on 786,432 rows, this takes 78.
__global__ void __launch_bounds__(RB) k_encode_bwd(Graph g, const float* __restrict__ g0,
                                                   float* __restrict__ part)
{
	__shared__ float red[WAVES][576];
	const int cg = threadIdx.x & 15, lane = threadIdx.x & 63, wave = wave_id();
	float acc[9][4];
#pragma unroll
	for(int v = 0; v < 9; v++)
#pragma unroll
		for(int i = 0; i < 4; i++) acc[v][i] = 0.f;
	const int stride = gridDim.x*(RB/16);
#pragma unroll 4
	for(int r = blockIdx.x*(RB/16) + (threadIdx.x >> 4); r < g.R; r += stride) {
		const f32x4 gv = *reinterpret_cast<const f32x4*>(g0 + (size_t)r*W + 4*cg);
		float x[FIN];
		node_x(g, r, x);
#pragma unroll
		for(int i = 0; i < 4; i++) {
#pragma unroll
			for(int f = 0; f < FIN; f++) acc[f][i] += x[f]*gv[i];
			acc[8][i] += gv[i];
		}
	}
#pragma unroll
	for(int f = 0; f < 9; f++)
#pragma unroll
		for(int i = 0; i < 4; i++) {
			float v = acc[f][i];
			v += __shfl_xor(v, 16);
			v += __shfl_xor(v, 32);
			if(lane < 16) red[wave][f*W + chan(4*cg) + i] = v;
		}
	__syncthreads();
	for(int i = threadIdx.x; i < 576; i += RB) {
		float v = 0.f;
		for(int w = 0; w < WAVES; w++) v += red[w][i];
		part[(size_t)blockIdx.x*576 + i] = v;
	}
}

// ------------------------------------------------------------------------------------------
// weight gradients on the MFMA units
// ------------------------------------------------------------------------------------------

constexpr int CH = 64;          // rows per LDS chunk
constexpr int WG_PART = 2*W*W + W + 2*W*W;

/// One layer's [dWu; dWv] = [hb | ab]^T dpre, dbu = sum dpre, [dWa | dWb] = hb^T dpq: the products'
/// depth is the rows, so chunks of 64 rows are transposed through LDS: a thread loads two channels
/// of 8 rows (a wave: whole rows) and writes 16 bytes per channel, the 16-byte units of a channel
/// exchanged by (channel/2) mod 8 and the two channels in the order of bit 3 of their pair, which
/// keeps writes and reads free of bank conflicts. The next chunk is loaded while this one is
/// multiplied. Wave w takes rows 16 w of dWu, dWv and [dWa | dWb].
///
/// Bound by HBM: 768 bytes per row. Two kernels that read h once each and transposed with
/// two-byte writes took 296 us on 786,432 rows, this takes 142 (604 MB, 83% of the copy rate).
__global__ void __launch_bounds__(RB, 2) k_wgrad(int R, int chunks_per_block,
                                                 const float* __restrict__ h,
                                                 const bf16_t* __restrict__ ab,
                                                 const bf16_t* __restrict__ dpre,
                                                 const bf16_t* __restrict__ dpq,
                                                 float* __restrict__ part)
{
	__shared__ __attribute__((aligned(16))) bf16_t T[5*W*CH];
	const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
	const int p = tid & 31, rg = tid >> 5, odd = (p >> 3) & 1;
	const f32x4 zero = f32x4{0.f, 0.f, 0.f, 0.f};
	f32x4 accu[2][4], accp[8], accb = zero;
#pragma unroll
	for(int j = 0; j < 4; j++) { accu[0][j] = zero; accu[1][j] = zero; }
#pragma unroll
	for(int j = 0; j < 8; j++) accp[j] = zero;
	const float one[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};
	const bf16x8 ones = to_frag(one);
	const int nchunk = (R + CH - 1)/CH;
	const int c_begin = blockIdx.x*chunks_per_block;
	const int c_end = min(c_begin + chunks_per_block, nchunk);
	float2 vh[8];
	unsigned vb[4][8];
	auto load = [&](int ch) {
#pragma unroll
		for(int i = 0; i < 8; i++) {
			const int r = ch*CH + 8*rg + i;
			const size_t rc = min(r, R - 1);
			vh[i] = *reinterpret_cast<const float2*>(h + rc*W + 2*p);
			vb[0][i] = *reinterpret_cast<const unsigned*>(ab + rc*W + 2*p);
			vb[1][i] = *reinterpret_cast<const unsigned*>(dpre + rc*W + 2*p);
			vb[2][i] = *reinterpret_cast<const unsigned*>(dpq + rc*2*W + 2*p);
			vb[3][i] = *reinterpret_cast<const unsigned*>(dpq + rc*2*W + W + 2*p);
		}
		if((ch + 1)*CH > R) {       // rows past the end count nothing
#pragma unroll
			for(int i = 0; i < 8; i++)
				if(ch*CH + 8*rg + i >= R) {
					vh[i] = make_float2(0.f, 0.f);
#pragma unroll
					for(int a = 0; a < 4; a++) vb[a][i] = 0u;
				}
		}
	};
	auto put = [&](int a, const unsigned* v) {      // v[i]: channels 2p (low), 2p + 1 of row 8 rg + i
		u32x4 lo, hi;
#pragma unroll
		for(int i = 0; i < 4; i++) {
			lo[i] = (v[2*i] & 0xFFFFu) | (v[2*i + 1] << 16);
			hi[i] = (v[2*i] >> 16) | (v[2*i + 1] & 0xFFFF0000u);
		}
		bf16_t* d = T + (W*a + 2*p)*CH + 8*(rg ^ (p & 7));
		*reinterpret_cast<u32x4*>(d + odd*CH) = odd ? hi : lo;
		*reinterpret_cast<u32x4*>(d + (1 - odd)*CH) = odd ? lo : hi;
	};
	auto frag = [&](int c16, int rgl) {
		const int c = c16 + (lane & 15);
		return *reinterpret_cast<const bf16x8*>(T + c*CH + 8*(rgl ^ ((c >> 1) & 7)));
	};
	if(c_begin < c_end) load(c_begin);
	for(int ch = c_begin; ch < c_end; ch++) {
		__syncthreads();
		{
			unsigned v[8];
#pragma unroll
			for(int i = 0; i < 8; i++) v[i] = pack2(vh[i].x, vh[i].y);
			put(0, v);
#pragma unroll
			for(int a = 0; a < 4; a++) put(1 + a, vb[a]);
		}
		__syncthreads();
		if(ch + 1 < c_end) load(ch + 1);
#pragma unroll
		for(int t = 0; t < CH/32; t++) {
			const int rgl = 4*t + (lane >> 4);
			const bf16x8 ah = frag(16*wave, rgl), aa = frag(W + 16*wave, rgl);
#pragma unroll
			for(int j = 0; j < 4; j++) {
				const bf16x8 b = frag(2*W + 16*j, rgl);
				accu[0][j] = mfma(ah, b, accu[0][j]);
				accu[1][j] = mfma(aa, b, accu[1][j]);
				if(j == wave) accb = mfma(ones, b, accb);
			}
#pragma unroll
			for(int j = 0; j < 8; j++) accp[j] = mfma(ah, frag(3*W + 16*j, rgl), accp[j]);
		}
	}
	float* out = part + (size_t)blockIdx.x*WG_PART;
	float* outp = out + 2*W*W + W;
#pragma unroll
	for(int i = 0; i < 4; i++) {
		const int k = 16*wave + 4*(lane >> 4) + i, kh = chan(k), n = lane & 15;
#pragma unroll
		for(int j = 0; j < 4; j++) {
			out[kh*W + 16*j + n] = accu[0][j][i];
			out[(W + k)*W + 16*j + n] = accu[1][j][i];
		}
#pragma unroll
		for(int j = 0; j < 8; j++) outp[kh*2*W + 16*j + n] = accp[j][i];
	}
	if(lane < 16) out[2*W*W + 16*wave + lane] = accb[0];
}

/// Sums `nblk` partials of `width` values into the flat gradient. A workgroup owns 16
/// consecutive values; its 16 lane groups each sum every 16th partial (in increasing order), and
/// the 16 group sums are added in group order, so the result is deterministic. Plain partials
/// go to off on, the last value to `extra` if given; k_wgrad's (weights) to their places among the
/// layer's weights, which start at off.
constexpr int RED_COLS = 16, RED_GROUPS = RB/RED_COLS;
__global__ void __launch_bounds__(RB) k_reduce(int nblk, int width, bool weights, int off,
                                               const float* __restrict__ part,
                                               float* __restrict__ grad, float* __restrict__ extra)
{
	__shared__ double sh[RB];
	const int c = threadIdx.x % RED_COLS, grp = threadIdx.x / RED_COLS;
	const int i = blockIdx.x*RED_COLS + c;
	double acc = 0.0;
	if(i < width)
		for(int b = grp; b < nblk; b += RED_GROUPS) acc += part[(size_t)b*width + i];
	sh[threadIdx.x] = acc;
	__syncthreads();
	if(grp != 0 || i >= width) return;
	double s = 0.0;
	for(int g = 0; g < RED_GROUPS; g++) s += sh[g*RED_COLS + c];
	int to = i;
	if(weights) {
		const int ip = i - (2*W*W + W);         // >= 0: [dWa | dWb]
		if(ip >= 0) to = (ip % (2*W) < W ? L_WA : L_WB - W) + ip/(2*W)*W + ip % (2*W);
		else if(i >= 2*W*W) to = L_BU + i - 2*W*W;
		else to = i < W*W ? L_WU + i : L_WV + i - W*W;
	} else if(extra && i == width - 1) {
		*extra = (float)s;
		return;
	}
	grad[off + to] = (float)s;
}

/// Adam (Kingma and Ba, 2015) on the fp32 master weights.
__global__ void __launch_bounds__(RB) k_adam(int n, float* __restrict__ w, float* __restrict__ m,
                                             float* __restrict__ v, const float* __restrict__ grad,
                                             float lr, float b1, float b2, float omb1, float omb2,
                                             float eps, float bc1, float bc2)
{
	const int i = blockIdx.x*RB + threadIdx.x;
	if(i >= n) return;
	const float gi = grad[i];
	const float mi = b1*m[i] + omb1*gi;
	const float vi = b2*v[i] + omb2*gi*gi;
	m[i] = mi;
	v[i] = vi;
	w[i] -= lr*(mi/bc1)/(sqrtf(vi/bc2) + eps);
}

/// Targets from conserved fields (see mpnn::targets on the host side).
__global__ void __launch_bounds__(RB) k_targets(int R, int N, const double* __restrict__ u,
                                                const double* __restrict__ pp, double gamma,
                                                float* __restrict__ t)
{
	const int r = blockIdx.x*RB + threadIdx.x;
	if(r >= R) return;
	const int gi = r / N;
	const double ca = pp[3*gi], sa = pp[3*gi + 1], pinf = pp[3*gi + 2];
	const double* q = u + (size_t)r*4;
	const double rho = q[0], vx = q[1]/rho, vy = q[2]/rho;
	const double p = (gamma - 1)*(q[3] - 0.5*rho*(vx*vx + vy*vy));
	float* o = t + (size_t)r*4;
	o[0] = (float)(rho - 1); o[1] = (float)(vx - ca); o[2] = (float)(vy - sa);
	o[3] = (float)(p/pinf - 1);
}

/// Conserved state from outputs, density and pressure floored at `floor` x freestream.
__global__ void __launch_bounds__(RB) k_warm(int R, int N, const float* __restrict__ y,
                                             const double* __restrict__ pp, double gamma,
                                             double floor, double* __restrict__ u)
{
	const int r = blockIdx.x*RB + threadIdx.x;
	if(r >= R) return;
	const int gi = r / N;
	const double ca = pp[3*gi], sa = pp[3*gi + 1], pinf = pp[3*gi + 2];
	const float* o = y + (size_t)r*4;
	const double rho = fmax(1.0 + (double)o[0], floor);
	const double vx = ca + (double)o[1], vy = sa + (double)o[2];
	const double p = fmax(1.0 + (double)o[3], floor)*pinf;
	double* q = u + (size_t)r*4;
	q[0] = rho; q[1] = rho*vx; q[2] = rho*vy; q[3] = p/(gamma - 1) + 0.5*rho*(vx*vx + vy*vy);
}

} // namespace mpnn

// ------------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------------

using namespace mpnn;

namespace {

double point_segment(double px, double py, double ax, double ay, double bx, double by)
{
	const double dx = bx - ax, dy = by - ay, ll = dx*dx + dy*dy;
	double t = ll > 0 ? ((px - ax)*dx + (py - ay)*dy)/ll : 0.0;
	t = std::min(1.0, std::max(0.0, t));
	const double qx = ax + t*dx - px, qy = ay + t*dy - py;
	return std::sqrt(qx*qx + qy*qy);
}

int blocks_for(size_t n) { return (int)((n + RB - 1)/RB); }

}

void mpnn_build_graph(const fvx_mesh_s& m, int wall_tag, MpnnGraphHost& gh)
{
	const int N = m.nelem;
	gh.N = N;
	gh.nbr.assign((size_t)N*4, -1);
	gh.rev.assign((size_t)N*4, -1);
	gh.invdeg.assign(N, 0.f);
	gh.stat.assign((size_t)N*NSTAT, 0.f);
	gh.edge.assign((size_t)N*16, 0.f);
	for(int c = 0; c < N; c++) {
		int deg = 0;
		for(int k = 0; k < 4; k++) {
			const int o = m.esuel[(size_t)c*4 + k];
			if(o >= 0 && o < N) { gh.nbr[(size_t)c*4 + k] = o; deg++; }
		}
		gh.invdeg[c] = deg > 0 ? (float)(1.0/deg) : 0.f;
	}
	for(int c = 0; c < N; c++)
		for(int k = 0; k < 4; k++) {
			const int j = gh.nbr[(size_t)c*4 + k];
			if(j < 0) continue;
			for(int kk = 0; kk < 4; kk++)
				if(gh.nbr[(size_t)j*4 + kk] == c
				   && m.elemface[(size_t)j*4 + kk] == m.elemface[(size_t)c*4 + k]) {
					gh.rev[(size_t)c*4 + k] = kk;
					break;
				}
			if(gh.rev[(size_t)c*4 + k] < 0)
				throw Error(FVX_ERR_INVALID, "mesh neighbour lists are not symmetric");
		}
	std::vector<int> wall;
	for(int b = 0; b < m.nbface; b++) if(m.btag[b] == wall_tag) wall.push_back(b);
	for(int c = 0; c < N; c++) {
		const double xc = m.rc[2*c], yc = m.rc[2*c + 1];
		const double r = std::hypot(xc - 0.5, yc);
		double dw = wall.empty() ? 1e4 : INFINITY;
		for(int b : wall) {
			const int p0 = m.bface[2*b], p1 = m.bface[2*b + 1];
			dw = std::min(dw, point_segment(xc, yc, m.coords[2*p0], m.coords[2*p0 + 1],
			                                m.coords[2*p1], m.coords[2*p1 + 1]));
		}
		double walladj = 0;
		for(int k = 0; k < 4; k++) {
			const int o = m.esuel[(size_t)c*4 + k];
			if(o >= N && m.btag[o - N] == wall_tag) walladj = 1;
		}
		float* s = &gh.stat[(size_t)c*NSTAT];
		s[0] = (float)((xc - 0.5)/(1 + r));
		s[1] = (float)(yc/(1 + r));
		s[2] = (float)(std::log1p(r)/std::log(51.0));
		s[3] = (float)(std::log10(dw + 1e-4)/2);
		s[4] = (float)(std::log10(std::sqrt(m.area[c]))/2);
		s[5] = (float)walladj;
		for(int k = 0; k < 4; k++) {
			const int j = gh.nbr[(size_t)c*4 + k];
			if(j < 0) continue;
			const double dx = m.rc[2*j] - xc, dy = m.rc[2*j + 1] - yc, L = std::hypot(dx, dy);
			float* e = &gh.edge[((size_t)c*4 + k)*4];
			e[0] = (float)(dx/L);
			e[1] = (float)(dy/L);
			e[2] = (float)std::log10(L/std::sqrt(m.area[c]));
			e[3] = (float)std::log(m.area[j]/m.area[c]);
		}
	}
}

void Mpnn::init(const fvx_mesh_s& m, int wall_tag, int max_graphs)
{
	mpnn_build_graph(m, wall_tag, host);
	N = host.N;
	cap = max_graphs;
	d_nbr.upload(host.nbr);
	d_rev.upload(host.rev);
	d_invdeg.upload(host.invdeg);
	d_stat.upload(host.stat);
	d_edge.upload(host.edge);
	const size_t R16 = ((size_t)cap*N + 15)/16*16;
	w.alloc(NPARAM); wq.alloc(NPARAM); am.alloc(NPARAM); av.alloc(NPARAM); grad.alloc(NPARAM);
	FVX_HIP(hipMemset(w.p, 0, NPARAM*sizeof(float)));
	FVX_HIP(hipMemset(am.p, 0, NPARAM*sizeof(float)));
	FVX_HIP(hipMemset(av.p, 0, NPARAM*sizeof(float)));
	frag.alloc((size_t)NL*4*FRAG_MAT);
	for(int l = 0; l < NL; l++) {
		h[l].alloc(R16*W);
		ab[l].alloc(R16*W);
		mmask[l].alloc(R16*8);
		if(l + 1 < NL) umask[l].alloc(R16*8);
	}
	for(int i = 0; i < 2; i++) {
		q[i].alloc(R16*W);
		da[i].alloc(R16*W);
		dpre[i].alloc(R16*W);
	}
	gpart.alloc(R16*W); dpq.alloc(R16*2*W);
	y.alloc(R16*FO);
	part.alloc((size_t)RED_BLOCKS*WG_PART);
	gfeat.alloc(2*(size_t)cap);
	pp.alloc(3*(size_t)cap);
	ids.alloc(cap);
	loss.alloc(1);
	dirty = true;
}

static Graph make_graph(const Mpnn& n, int G)
{
	Graph g;
	g.N = n.N; g.R = G*n.N;
	g.nbr = n.d_nbr.p; g.rev = n.d_rev.p; g.invdeg = n.d_invdeg.p; g.stat = n.d_stat.p;
	g.edge = n.d_edge.p; g.gfeat = n.gfeat.p;
	return g;
}

void Mpnn::set_points(int G, const double* mach, const double* aoa, double gamma, hipStream_t s)
{
	if(G < 1 || G > cap) throw Error(FVX_ERR_INVALID, "graph count outside [1, max_graphs]");
	this->gamma = gamma;
	npoints = G;
	hgf.resize(2*(size_t)G);
	hpp.resize(3*(size_t)G);
	for(int i = 0; i < G; i++) {
		if(!(mach[i] > 0) || !std::isfinite(mach[i]) || !std::isfinite(aoa[i]))
			throw Error(FVX_ERR_INVALID, "invalid Mach number or angle of attack");
		const double a = aoa[i];
		hgf[2*i] = (float)(4.0*(mach[i] - 0.5));
		hgf[2*i + 1] = (float)(a*(180.0/M_PI)/5.0);
		hpp[3*i] = std::cos(a); hpp[3*i + 1] = std::sin(a);
		hpp[3*i + 2] = 1.0/(gamma*mach[i]*mach[i]);
	}
	FVX_HIP(hipMemcpyAsync(gfeat.p, hgf.data(), hgf.size()*sizeof(float), hipMemcpyHostToDevice, s));
	FVX_HIP(hipMemcpyAsync(pp.p, hpp.data(), hpp.size()*sizeof(double), hipMemcpyHostToDevice, s));
}

void Mpnn::pack(hipStream_t s)
{
	if(!dirty) return;
	const int n = std::max(NPARAM, NL*4*FRAG_MAT);
	k_pack<<<blocks_for(n), RB, 0, s>>>(w.p, wq.p, frag.p);
	FVX_HIP(hipGetLastError());
	dirty = false;
}

/// Workgroups of the row-tile kernels: as many as are resident at once (LDS: 3 a compute unit).
static int tile_grid(int R) { return std::max(1, std::min(TILE_BLOCKS, ((R + 15)/16 + WAVES - 1)/WAVES)); }

void Mpnn::forward(int G, const float* targets, float* yout, hipStream_t s)
{
	pack(s);
	const Graph g = make_graph(*this, G);
	const int R = g.R, nt = (R + 15)/16, nb = tile_grid(R);
	const double inv = 1.0/((double)R*FO);
	k_embed<<<nb, RB, 0, s>>>(g, nt, wq.p, frag.p + M_PQ*FRAG_MAT, h[0].p, q[0].p);
	for(int l = 0; l < NL; l++) {
		const bf16_t* fl = frag.p + (size_t)l*4*FRAG_MAT;
		const bool last = l + 1 == NL;
		auto run = [&](auto kernel) {
			kernel<<<nb, RB, 0, s>>>(g, nt, h[l].p, q[l & 1].p, wq.p + OFF_L0 + l*LSZ,
				fl + M_PQ*FRAG_MAT, fl + M_UPD*FRAG_MAT, fl + (last ? M_BUPD : 4 + M_PQ)*FRAG_MAT, wq.p,
				last ? nullptr : h[l + 1].p, q[(l + 1) & 1].p, ab[l].p, last ? nullptr : umask[l].p, mmask[l].p,
				yout, targets, ids.p, inv, dpre[l & 1].p, gpart.p, da[l & 1].p, part.p);
		};
		if(!last) { if(targets) run(k_layer<true, false>); else run(k_layer<false, false>); }
		else if(targets) run(k_layer<true, true>);
		else run(k_layer<false, true>);
	}
	FVX_HIP(hipGetLastError());
}

void Mpnn::predict(int G, float* yout, hipStream_t s)
{
	forward(G, nullptr, yout, s);
}

void Mpnn::gradient(int G, const float* targets, const int* sample_ids, hipStream_t s)
{
	for(int i = 0; i < G; i++)
		if(sample_ids[i] < 0) throw Error(FVX_ERR_INVALID, "negative sample index");
	hids.assign(sample_ids, sample_ids + G);
	FVX_HIP(hipMemcpyAsync(ids.p, hids.data(), G*sizeof(int), hipMemcpyHostToDevice, s));
	forward(G, targets, nullptr, s);
	const Graph g = make_graph(*this, G);
	const int R = g.R, nt = (R + 15)/16, nb = tile_grid(R);
	auto reduce = [&](int nblk, int width, bool weights, int off, float* extra) {
		k_reduce<<<(width + RED_COLS - 1)/RED_COLS, RB, 0, s>>>(nblk, width, weights, off, part.p,
		                                                       grad.p, extra);
	};
	reduce(nb, 261, false, OFF_WDEC, loss.p);
	const int nchunk = (R + CH - 1)/CH;
	const int cpb = (nchunk + RED_BLOCKS - 1)/RED_BLOCKS;
	const int nwb = (nchunk + cpb - 1)/cpb;
	// da[l & 1] and dpre[l & 1] hold layer l's; the backward pass of a layer leaves those of the one
	// before it
	for(int l = NL - 1; l >= 0; l--) {
		const bf16_t* fl = frag.p + (size_t)l*4*FRAG_MAT;
		const int base = OFF_L0 + l*LSZ, a = l & 1, b = 1 - a;
		if(l > 0)
			k_layer_bwd<false><<<nb, RB, 0, s>>>(g, nt, da[a].p, mmask[l].p, fl + M_BPQ*FRAG_MAT,
				fl + (M_BUPD - 4)*FRAG_MAT, umask[l - 1].p, dpq.p, gpart.p, dpre[b].p, da[b].p, part.p);
		else
			k_layer_bwd<true><<<nb, RB, 0, s>>>(g, nt, da[a].p, mmask[l].p, fl + M_BPQ*FRAG_MAT, nullptr,
				nullptr, dpq.p, gpart.p, nullptr, nullptr, part.p);
		reduce(nb, 320, false, base + L_WE, nullptr);
		k_wgrad<<<nwb, RB, 0, s>>>(R, cpb, h[l].p, ab[l].p, dpre[a].p, dpq.p, part.p);
		reduce(nwb, WG_PART, true, base, nullptr);
	}
	k_encode_bwd<<<RED_BLOCKS, RB, 0, s>>>(g, gpart.p, part.p);
	reduce(RED_BLOCKS, 576, false, OFF_WENC, nullptr);
	FVX_HIP(hipGetLastError());
}

void Mpnn::adam_step(double lr, hipStream_t s)
{
	step++;
	const double b1 = 0.9, b2 = 0.999;
	const float bc1 = (float)(1.0 - std::pow(b1, step)), bc2 = (float)(1.0 - std::pow(b2, step));
	k_adam<<<blocks_for(NPARAM), RB, 0, s>>>(NPARAM, w.p, am.p, av.p, grad.p, (float)lr, (float)b1,
	                                         (float)b2, (float)(1 - b1), (float)(1 - b2), 1e-8f,
	                                         bc1, bc2);
	FVX_HIP(hipGetLastError());
	dirty = true;
}

void Mpnn::targets(int G, const double* u, float* t, hipStream_t s)
{
	k_targets<<<blocks_for((size_t)G*N), RB, 0, s>>>(G*N, N, u, pp.p, gamma, t);
	FVX_HIP(hipGetLastError());
}

void Mpnn::warm(int G, double floor, double* u, hipStream_t s)
{
	predict(G, y.p, s);
	k_warm<<<blocks_for((size_t)G*N), RB, 0, s>>>(G*N, N, y.p, pp.p, gamma, floor, u);
	FVX_HIP(hipGetLastError());
}

} // namespace fvx
