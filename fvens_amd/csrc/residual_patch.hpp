/* residual_patch.hpp -- gradients, limiter, face fluxes and cell sums of a second-order residual in
 * one launch.
 *
 * Reference semantics: GradientScheme::compute_gradients, the limiters and
 * FlowFV::compute_residual, as in spatial.hip (k_gradients) and flux_kernel.hpp; every value is
 * formed by the same operations in the same order, so the result is bitwise that of the separate
 * passes.
 *
 * A workgroup owns a patch of neighbouring cells whose faces make at most 256 tasks (flux_wave.hpp
 * explains tasks) and also lists the halo, the patch's outer neighbours, and beyond it the cells
 * and boundary faces whose states the gradients of patch and halo need:
 *   1. primitive states of all of them to LDS, ghost states formed in place, and the centres of
 *      patch and halo;
 *   2. the (limited) gradients of patch and halo, two lanes per cell, each visiting two of its faces;
 *   3. one face task per lane from the states and gradients in LDS, its results to LDS;
 *   4. each own cell adds its four slots.
 * Halo gradients are computed by several patches: 1.28x the gradient work on 4,608 cells in RCM
 * order, 1.41x on 98,304, 1.47x on 1,572,864 in Hilbert order, 1.53x on 262,144 viscous
 * quadrilaterals (where the order is compact by rows, patches of consecutive cells are strips:
 * 2.3x on the 4,608 cells as generated). That costs less
 * than writing and reading them (160 bytes a cell with the second read of the state, of 408) and
 * two more launches: 1,572,864 cells in Hilbert order (HLLC, limited) 207 -> 176 us, 16 instances
 * of 98,304 cells (Roe, limited) 197 -> 153, 262,144 cells viscous MUSCL 78 -> 53, 4,608 cells 20
 * -> 13. Bound by HBM (1,572,864 cells: 660 MB, 77% of the copy rate) and FP64 issue (56% of the
 * time). Four waves per SIMD for Roe, which would spill at five (16 instances 145 against 149 us
 * in a row), five for the other fluxes (HLLC on 1,572,864 cells 175 against 186); viscous three.
 * Larger patches would have fewer halo cells, but more than 256 tasks, one per lane. A patch cell's
 * midpoint offsets from its faces' records instead of the table save 10% of the traffic, but the
 * gradients then wait for the records: 177 -> 200 us.
 */
#ifndef FVX_RESIDUAL_PATCH_HPP
#define FVX_RESIDUAL_PATCH_HPP

#include "flux_kernel.hpp"

namespace fvx {

constexpr unsigned PATCH_NONE = 0xffff;      // an unused slot

/// p ? b : a of values (a conditional on array elements is turned into an indexed array in scratch)
__device__ __forceinline__ double pick(int p, double a, double b) { return p ? b : a; }

template <int FLUX, int LIM, int MODE, bool VISC>
__global__ __launch_bounds__(PATCH_TASKS, VISC ? 3 : FLUX == 0 ? 4 : 5)
void k_residual_patch(int ncell, int nw, int ns, const double* __restrict__ u, PatchTables pt,
                      const double* __restrict__ soff,
                      const double* __restrict__ gcoef, const double* __restrict__ eps2,
                      const FaceGeom* __restrict__ fgeom, const double* __restrict__ centre,
                      const double* __restrict__ area, const int* __restrict__ bcid,
                      const GasParams* __restrict__ gpa, const BCTable* __restrict__ bta,
                      const BatchArg ba, double* __restrict__ res, double* __restrict__ dt,
                      const int getdt, const int xcd)
{
	const long I = ba.list ? ba.list[blockIdx.y] : 0;
	if(I < 0) return;                     // a retired slot of a compacted list
	const GasParams& gp = gpa[I];
	const BCTable& bt = *bta;
	u += I*4L*ncell;
	res += I*4L*ncell;
	if(dt) dt += I*(long)ncell;
	extern __shared__ double sm[];        // [nw] 4 w; [ns] 2 centre, 8 gradient
	double* const sw = sm;
	double* const sx = sm + 4*nw;
	double* const sg = sx + 2*ns;
	const int g = xcd_block(xcd), tid = threadIdx.x;
	const double igm1 = 1.0/gp.gm1;
	const PatchGroup G4 = pt.groups[g];
	const int* list = pt.cells + G4.list;
	const int nl = G4.nlist, nown = G4.nown;
	const int f = pt.face[(size_t)g*PATCH_TASKS + tid];
	const unsigned lr = pt.sides[(size_t)g*PATCH_TASKS + tid];
	for(int i = tid; i < G4.nstate; i += PATCH_TASKS) {
		const int c = list[i];
		double uc[4], w[4];
		if(c >= 0) load4(u + 4*c, uc);
		else {
			const FaceGeom F = fgeom[-1 - c];  // boundary faces are numbered first
			const double n[2] = { F.nx, F.ny };
			double ui[4];
			load4(u + 4*F.left, ui);
			ghost_state(gp, bt, bcid[-1 - c], ui, n, uc);
		}
		if(i < nl) {
			const double2 x = reinterpret_cast<const double2*>(centre)[c];
			sx[i] = x.x;
			sx[ns + i] = x.y;
		}
		prim_lean(gp, uc, w);
		for(int v = 0; v < 4; v++) sw[v*nw + i] = w[v];
	}
	__syncthreads();

	for(int i = tid >> 1; i < nl; i += PATCH_TASKS/2) {
		const int p = tid & 1, c = list[i];
		const ushort2 lc2 = reinterpret_cast<const ushort2*>(pt.local)[2*(G4.local + i) + p];
		const unsigned lc[2] = { lc2.x, lc2.y };
		const double2* cf = reinterpret_cast<const double2*>(gcoef) + 4*c + 2*p;
		const double2 cfv[2] = { cf[0], cf[1] };
		double2 off[2] = { make_double2(0, 0), make_double2(0, 0) };
		double e2 = 0.0;
		if constexpr(LIM > 0) {
			const double2* so = reinterpret_cast<const double2*>(soff) + 4*c + 2*p;
			off[0] = so[0];
			off[1] = so[1];
			if constexpr(LIM == 1) e2 = eps2[c];
		}
		double wi[4];
		for(int v = 0; v < 4; v++) wi[v] = sw[v*nw + i];
		double d[8] = {0, 0, 0, 0, 0, 0, 0, 0};
		double dmax[4] = {0, 0, 0, 0}, dmin[4] = {0, 0, 0, 0};
#pragma unroll
		for(int k = 0; k < 2; k++) {
			if(lc[k] == PATCH_NONE) continue;
			double wj[4];
			for(int v = 0; v < 4; v++) wj[v] = sw[v*nw + lc[k]];
			for(int v = 0; v < 4; v++) {
				const double dw = wj[v] - wi[v];
				d[2*v] += cfv[k].x*dw;
				d[2*v+1] += cfv[k].y*dw;
				if constexpr(LIM > 0) { dmax[v] = fmax(dmax[v], dw); dmin[v] = fmin(dmin[v], dw); }
			}
		}
		for(int k = 0; k < 8; k++) d[k] = pair_sum(d[k]);
		// lane p finishes the variables 2p and 2p + 1
		if constexpr(LIM == 0) {
			for(int k = 0; k < 4; k++) sg[(4*p + k)*ns + i] = pick(p, d[k], d[4 + k]);
		} else {
			double bn[4], bd[4];
			for(int v = 0; v < 4; v++) {
				const double mx = pair_max(dmax[v]), mn = pair_min(dmin[v]);
				bn[v] = bd[v] = 1.0;            // the smallest ratio so far, as N / D (k_gradients)
				for(int k = 0; k < 2; k++) {
					if(lc[k] == PATCH_NONE) continue;
					double uf = wi[v];
					uf += d[2*v]*off[k].x;
					uf += d[2*v+1]*off[k].y;
					const double dm = uf - wi[v];
					double pn, pd;
					if constexpr(LIM == 1) {
						const double dp = dm < 0 ? mn : mx;
						pn = dp*dp + 2*dp*dm + e2;
						pd = dp*dp + dp*dm + 2*dm*dm + e2;
					} else {
						if(dm > 0) { pn = mx; pd = dm; }
						else if(dm < 0) { pn = -mn; pd = -dm; }
						else { pn = 1.0; pd = 1.0; }
					}
					if(pn*bd[v] < bn[v]*pd) { bn[v] = pn; bd[v] = pd; }
				}
			}
			for(int j = 0; j < 2; j++) {
				// own candidate, and the other lane's for the same variable; the slots 2, 3 win if smaller
				const double on = dpp_d<DPP_XOR1>(pick(p, bn[2 + j], bn[j]));
				const double od = dpp_d<DPP_XOR1>(pick(p, bd[2 + j], bd[j]));
				double tn = pick(p, bn[j], bn[2 + j]), td = pick(p, bd[j], bd[2 + j]);
				if(p == 0) { if(on*td < tn*od) { tn = on; td = od; } }
				else { if(!(tn*od < on*td)) { tn = on; td = od; } }
				const double phi = tn/td;
				sg[(4*p + 2*j)*ns + i] = phi*pick(p, d[2*j], d[4 + 2*j]);
				sg[(4*p + 2*j + 1)*ns + i] = phi*pick(p, d[2*j + 1], d[5 + 2*j]);
			}
		}
	}
	__syncthreads();

	double FL[4], radL = 0.0, radR = 0.0;
	if(f >= 0) {
		const FaceGeom G = fgeom[f];
		const double n[2] = { G.nx, G.ny };
		const bool bnd = G.right < 0;
		const int l = lr & 0xffff, r = lr >> 16;  // r: the ghost's state entry for a boundary face
		double wL[4], wR[4], gL[8], gR[8], xL[2], xR[2];
		int bc = 0;
		for(int v = 0; v < 4; v++) { wL[v] = sw[v*nw + l]; wR[v] = sw[v*nw + r]; }
		const int rg = bnd ? l : r;
		for(int k = 0; k < 8; k++) gL[k] = sg[k*ns + l];
		for(int k = 0; k < 8; k++) gR[k] = sg[k*ns + rg];
		xL[0] = sx[l]; xL[1] = sx[ns + l];
		xR[0] = sx[rg]; xR[1] = sx[ns + rg];
		if(bnd) {
			bc = bcid[-1 - G.right];
			xR[0] = 2.0*G.mx - xL[0]; xR[1] = 2.0*G.my - xL[1];
		}
		FaceState A, B;
		double q[4];
		if constexpr(MODE == 1) {
			const double dx = G.mx - xL[0], dy = G.my - xL[1];
			for(int k = 0; k < 4; k++) q[k] = wL[k] + gL[2*k]*dx + gL[2*k+1]*dy;
			A = fs_prim(gp, q, n, igm1);
			if(!bnd) {
				const double ex = G.mx - xR[0], ey = G.my - xR[1];
				for(int k = 0; k < 4; k++) q[k] = wR[k] + gR[2*k]*ex + gR[2*k+1]*ey;
				B = fs_prim(gp, q, n, igm1);
			}
		} else {
			double q2[4];
			muscl_states(wL, wR, gL, gR, xR[0] - xL[0], xR[1] - xL[1], bnd, q, q2);
			A = fs_prim(gp, q, n, igm1);
			if(!bnd) B = fs_prim(gp, q2, n, igm1);
		}
		if(bnd) {
			const double UL[4] = { A.r, A.mx, A.my, A.E };
			double UG[4];
			ghost_state(gp, bt, bc, UL, n, UG);
			B = fs_cons(gp, UG, n);
		}
		fs_num_flux<FLUX>(gp, A, B, n, FL);
		if constexpr(VISC) {
			double vf[4];
			viscous_flux(gp, n, xL, xR, wL, 1.0/wL[0], wR, 1.0/wR[0], gL, gR, A, B, vf);
			for(int k = 0; k < 4; k++) FL[k] += vf[k];
		}
		for(int v = 0; v < 4; v++) FL[v] = G.len*FL[v];
		radL = face_radius<VISC>(gp, A, G.len, area, G.left);
		if(!VISC || !bnd) radR = face_radius<VISC>(gp, B, G.len, area, G.right);
	}
	__syncthreads();
	double* const sp = sg;                // the gradients' place, ns >= 192: 6 x 256 values
	if(f >= 0) {
		for(int v = 0; v < 4; v++) sp[v*PATCH_TASKS + tid] = FL[v];
		sp[4*PATCH_TASKS + tid] = radL;
		sp[5*PATCH_TASKS + tid] = radR;
	}
	__syncthreads();

	if(tid < nown) {
		const int c = list[tid];
		const ushort4 cs = pt.slots[G4.slots + tid];
		const unsigned code[4] = { cs.x, cs.y, cs.z, cs.w };
		double s[4][5];
		for(int k = 0; k < 4; k++) {
			if(code[k] == PATCH_NONE) {
				for(int v = 0; v < 5; v++) s[k][v] = 0.0;
				continue;
			}
			const int task = (int)(code[k] >> 1), side = (int)(code[k] & 1u);
			for(int v = 0; v < 4; v++) {
				const double F = sp[v*PATCH_TASKS + task];
				s[k][v] = side ? F : -F;
			}
			s[k][4] = sp[(4 + side)*PATCH_TASKS + task];
		}
		double rv[4];
		load4(res + 4*c, rv);
		for(int v = 0; v < 4; v++) rv[v] += (s[0][v] + s[1][v]) + (s[2][v] + s[3][v]);
		store4(res + 4*c, rv);
		if(getdt) dt[c] = area[c]/((s[0][4] + s[1][4]) + (s[2][4] + s[3][4]));
	}
}

}
#endif
