/* jacobian.hip -- first-order approximate Jacobian assembly (Spatial::assemble_jacobian).
 *
 * Reference semantics: Spatial::assemble_jacobian (src/spatial/aspatial.cpp:242-340) with
 * FlowFV::compute_local_jacobian_interior / _boundary (src/spatial/flow_spatial.cpp:818-875):
 * the Jacobian of the FIRST-ORDER residual evaluated at the cell-centred states. For an interior
 * face with left cell L (lower index) and right cell R, F = F(u_L, u_R) times the face length
 * leaves L and enters R, so the row of L gains +len dF/du_L on its diagonal and +len dF/du_R in
 * column R, and the row of R gains -len dF/du_R on its diagonal and -len dF/du_L in column L.
 * A boundary face adds len (dF/du_L + dF/du_g du_g/du_L) to the diagonal, with the ghost state
 * and its Jacobian from FlowBC::computeGhostStateAndJacobian (src/spatial/abc.cpp).
 *
 * Flux Jacobians (InviscidFlux::get_jacobian): Roe (anumericalflux.cpp:736-965), HLLC
 * (:1230-1397) and AUSM (:317-472) are differentiated exactly here with forward-mode duals
 * through the same templated flux code the residual uses; LLF (:65-107) and HLL (:1012-1061)
 * use the reference's frozen-eigenvalue / frozen-speed forms. The viscous part is the
 * thin-layer flux of flow_spatial.cpp:397-446 / aspatial.cpp:207-240, differentiated exactly.
 *
 * Storage ("slot blocks"): vals[cell][slot][4][4] row-major, slot 0 the diagonal block and slot
 * 1+k the block of the neighbour across local face k (nbr[cell][k]); slots without an interior
 * neighbour hold zeros. Each cell's quad of lanes evaluates its own faces (each interior face
 * twice, once from each side, from identical canonical data), so assembly needs no atomics and
 * is bitwise reproducible.
 */
#include "fvx_internal.hpp"
#include "gas.hpp"
#include "dual.hpp"
#include "wave.hpp"

namespace fvx {

using D4 = Dual<4>;
using D1 = Dual<1>;

/// Cells of a workgroup of `block` threads (k_jacobian).
__host__ __device__ constexpr int jac_cells(int block) { return block == 64 ? 16 : block/8; }

/// Thin-layer viscous flux of two cell states: face gradient (q_R - q_L)/|dr| along the unit
/// centre-to-centre vector, q = (rho, vx, vy, T) (viscousphysics.cpp:124-246).
template <class TA, class TB, class T = FaceScalar<TA, TB>>
__device__ __forceinline__ void thinlayer_flux(const GasParams& gp, const double* n,
                                               const double* xl, const double* xr,
                                               const TA* ul, const TB* ur, T* vf)
{
	TA wl[4];
	TB wr[4];
	wl[0] = ul[0]; wl[1] = ul[1]/ul[0]; wl[2] = ul[2]/ul[0];
	wl[3] = pressure(gp, ul)/ul[0]*gp.gM2;
	wr[0] = ur[0]; wr[1] = ur[1]/ur[0]; wr[2] = ur[2]/ur[0];
	wr[3] = pressure(gp, ur)/ur[0]*gp.gM2;
	double dr[2] = { xr[0] - xl[0], xr[1] - xl[1] };
	const double dist = sqrt(dr[0]*dr[0] + dr[1]*dr[1]);
	dr[0] /= dist; dr[1] /= dist;
	T grad[2][4];
	for(int i = 0; i < 4; i++) {
		const T corr = (wr[i] - wl[i])/dist;
		grad[0][i] = corr*dr[0];
		grad[1][i] = corr*dr[1];
	}
	T mu;
	if(gp.constvisc) mu = T(1.0/gp.Reinf);
	else mu = 0.5*(sutherland(gp, wl[3]) + sutherland(gp, wr[3]));
	const T kd = mu/(gp.Minf*gp.Minf*gp.gm1*gp.Pr);
	const T ldiv = 2.0/3.0*mu*(grad[0][1] + grad[1][2]);
	T s[2][2];
	for(int i = 0; i < 2; i++) {
		for(int j = 0; j < 2; j++) s[i][j] = mu*(grad[i][j+1] + grad[j][i+1]);
		s[i][i] -= ldiv;
	}
	vf[0] = T(0.0);
	vf[1] = -(s[0][0]*n[0] + s[0][1]*n[1]);
	vf[2] = -(s[1][0]*n[0] + s[1][1]*n[1]);
	const T va0 = 0.5*(wl[1] + wr[1]), va1 = 0.5*(wl[2] + wr[2]);
	T e = T(0.0);
	for(int i = 0; i < 2; i++) {
		const T comp = s[i][0]*va0 + s[i][1]*va1 + kd*grad[i][3];
		e -= comp*n[i];
	}
	vf[3] = e;
}

/// Ghost state and column j of du_g/du_in. Every kind except the isothermal wall is the exact
/// derivative of ghost_state (abc.cpp:86-140, 201-210, 228-262, 282-305, 425-437), obtained with
/// duals; the isothermal wall uses the reference's own linearisation, including its ghost
/// energy at the wall temperature (abc.cpp:371-409).
__device__ __forceinline__ void ghost_column(const GasParams& gp, const BCTable& bt, int bc,
                                             const double* ui, const double* n, int j,
                                             double* ug, double* dug)
{
	if(bt.kind[bc] == 6) {
		const double v0 = bt.v0[bc], v1 = bt.v1[bc];
		const double tm = v0*ui[0];
		ug[0] = ui[0];
		ug[1] = 2.0*tm*n[1] - ui[1];
		ug[2] = -2.0*tm*n[0] - ui[2];
		const double m2 = ug[1]*ug[1] + ug[2]*ug[2];
		const double ir2 = 1.0/(ui[0]*ui[0]);
		const double vmag2 = m2*ir2;
		const double coeff = 1.0/(gp.g*gp.gm1*gp.Minf*gp.Minf);
		ug[3] = ui[0]*(v1*coeff + 0.5*vmag2);
		const double dv0 = -2.0*m2*ir2/ui[0];
		dug[0] = j == 0 ? 1.0 : 0.0;
		dug[1] = j == 0 ? 2.0*v0*n[1] : j == 1 ? -1.0 : 0.0;
		dug[2] = j == 0 ? -2.0*v0*n[0] : j == 2 ? -1.0 : 0.0;
		dug[3] = j == 0 ? coeff*v1 + 0.5*(vmag2 + ui[0]*dv0) : j == 1 ? ui[0]*0.5*(-ug[1]*ir2)
		         : j == 2 ? ui[0]*0.5*(-ug[2]*ir2) : 0.0;
		return;
	}
	D1 a[4], g[4];
#pragma unroll
	for(int k = 0; k < 4; k++) { a[k] = D1(ui[k]); a[k].d[0] = k == j ? 1.0 : 0.0; }
	ghost_state(gp, bt, bc, a, n, g);
#pragma unroll
	for(int i = 0; i < 4; i++) { ug[i] = g[i].v; dug[i] = g[i].d[0]; }
}

/// dF/du of the analytic directional flux (aphysics_defs.hpp:13-23), by duals.
__device__ __forceinline__ void phys_flux_jacobian(const GasParams& gp, const double* u,
                                                   const double* n, double* A)
{
	D4 a[4], f[4];
	for(int k = 0; k < 4; k++) { a[k] = D4(u[k]); a[k].d[k] = 1.0; }
	const D4 vn = (a[1]*n[0] + a[2]*n[1])/a[0];
	phys_flux(a, n, vn, pressure(gp, a), f);
	for(int i = 0; i < 4; i++)
		for(int j = 0; j < 4; j++) A[i*4+j] = f[i].d[j];
}

/// Derivative dF/du of one side (SIDE 0: left, 1: right) of the Jacobian flux (plus the
/// thin-layer viscous flux when VISC) at cell-centred states, row-major. Only the side's own
/// variables are duals.
template <int FLUX, bool VISC, int SIDE>
__device__ __forceinline__ void side_jacobian(const GasParams& gp, const double* n,
                                              const double* xl, const double* xr,
                                              const double* ul, const double* ur, double* J)
{
	D4 s4[4], f[4];
	Val o[4];
	const double* us = SIDE == 0 ? ul : ur;
	const double* uo = SIDE == 0 ? ur : ul;
#pragma unroll
	for(int k = 0; k < 4; k++) { s4[k] = D4(us[k]); s4[k].d[k] = 1.0; o[k] = Val(uo[k]); }
	if constexpr(FLUX == 2 || FLUX == 3) {
		phys_flux_jacobian(gp, us, n, J);
		const SideVars<double> a = side_vars(gp, ul, n), b = side_vars(gp, ur, n);
		const double ca = sqrt(gp.g*a.p/ul[0]), cb = sqrt(gp.g*b.p/ur[0]);
		double w, d;               // J <- w J + d I
		if constexpr(FLUX == 3) {
			const double ea = fabs(a.vn) + ca, eb = fabs(b.vn) + cb;
			const double eig = ea >= eb ? ea : eb;
			w = 0.5; d = SIDE == 0 ? 0.5*eig : -0.5*eig;
		} else {
			const RoeAvg<double> m = roe_avg(gp, ul, ur, n, a, b);
			double sl, sr;
			einfeldt(a.vn, ca, b.vn, cb, m, sl, sr);
			const double sr0 = sr > 0.0 ? 0.0 : sr, sl0 = sl > 0.0 ? 0.0 : sl;
			const double t1 = (sr0 - sl0)/(sr - sl), t2 = 1.0 - t1;
			const double t3 = 0.5*(sr*fabs(sl) - sl*fabs(sr))/(sr - sl);
			w = SIDE == 0 ? t2 : t1; d = SIDE == 0 ? t3 : -t3;
		}
#pragma unroll
		for(int k = 0; k < 16; k++) J[k] *= w;
#pragma unroll
		for(int i = 0; i < 4; i++) J[i*5] += d;
		if constexpr(VISC) {
			if constexpr(SIDE == 0) thinlayer_flux(gp, n, xl, xr, s4, o, f);
			else thinlayer_flux(gp, n, xl, xr, o, s4, f);
#pragma unroll
			for(int i = 0; i < 4; i++)
#pragma unroll
				for(int j = 0; j < 4; j++) J[i*4+j] += f[i].d[j];
		}
	} else {
		if constexpr(SIDE == 0) num_flux<FLUX>(gp, s4, o, n, f);
		else num_flux<FLUX>(gp, o, s4, n, f);
		if constexpr(VISC) {
			D4 vf[4];
			if constexpr(SIDE == 0) thinlayer_flux(gp, n, xl, xr, s4, o, vf);
			else thinlayer_flux(gp, n, xl, xr, o, s4, vf);
#pragma unroll
			for(int k = 0; k < 4; k++) f[k] += vf[k];
		}
#pragma unroll
		for(int i = 0; i < 4; i++)
#pragma unroll
			for(int j = 0; j < 4; j++) J[i*4+j] = f[i].d[j];
	}
}

/// Column j of the total derivative d/du_L of F(u_L, u_g(u_L)) at a boundary face.
template <int FLUX, bool VISC>
__device__ __forceinline__ void boundary_column(const GasParams& gp, const BCTable& bt, int bc,
                                                const double* n, const double* xl,
                                                const double* xg, const double* ul, int j,
                                                double* col)
{
	double ug[4], dug[4];
	ghost_column(gp, bt, bc, ul, n, j, ug, dug);
	if constexpr(FLUX == 2 || FLUX == 3) {
		double JL[16], JR[16];
		side_jacobian<FLUX, VISC, 0>(gp, n, xl, xg, ul, ug, JL);
		side_jacobian<FLUX, VISC, 1>(gp, n, xl, xg, ul, ug, JR);
#pragma unroll
		for(int i = 0; i < 4; i++) {
			double s = 0.0;
#pragma unroll
			for(int k = 0; k < 4; k++) s += JR[i*4+k]*dug[k];
			double v = JL[i*4];
#pragma unroll
			for(int k = 1; k < 4; k++) v = j == k ? JL[i*4+k] : v;
			col[i] = v + s;
		}
	} else {
		D1 a[4], g[4], f[4];
#pragma unroll
		for(int i = 0; i < 4; i++) {
			a[i] = D1(ul[i]); a[i].d[0] = i == j ? 1.0 : 0.0;
			g[i] = D1(ug[i]); g[i].d[0] = dug[i];
		}
		num_flux<FLUX>(gp, a, g, n, f);
		if constexpr(VISC) {
			D1 vf[4];
			thinlayer_flux(gp, n, xl, xg, a, g, vf);
#pragma unroll
			for(int k = 0; k < 4; k++) f[k] += vf[k];
		}
#pragma unroll
		for(int i = 0; i < 4; i++) col[i] = f[i].d[0];
	}
}

template <class VT> __device__ __forceinline__ void store_row(VT* p, const double* v);
template <> __device__ __forceinline__ void store_row<double>(double* p, const double* v)
{
	reinterpret_cast<double2*>(p)[0] = make_double2(v[0], v[1]);
	reinterpret_cast<double2*>(p)[1] = make_double2(v[2], v[3]);
}
template <> __device__ __forceinline__ void store_row<float>(float* p, const double* v)
{
	*reinterpret_cast<float4*>(p) = make_float4((float)v[0], (float)v[1], (float)v[2],
	                                            (float)v[3]);
}

/// A pair of waves per 16 cells: the quad of lanes of a cell owns its four faces in both, one
/// wave differentiates the faces by their left states, the other by their right ones (a
/// workgroup of one wave does both in turn), and the derivatives meet in LDS, from where the
/// rows are written. When dt is given the pseudo-time term area/(cfl dt) is added to
/// the diagonal and stored in dtm (SteadyBackwardEulerSolver::addPseudoTimeTerm,
/// src/ode/aodesolver.cpp:300-329).
///
/// Bound by FP64 VALU work and its latency: ~1,000 instructions a face and side at two waves per
/// SIMD (204-228 registers; viscous up to 255, HLL and LLF spill 44 bytes a lane: 60 and 55 us on
/// 98,304 cells, 75 and 71 with both sides on a lane). One lane differentiating both sides in turn, all variables duals,
/// needed 290-380 registers and spilled. Assembly on 98,304 cells, FP64, workgroups of 64: Roe
/// 120 -> 43 us, HLLC 74 -> 44 us; 4,608 cells, workgroups of 256: Roe 25 -> 12 us, HLLC 19 -> 12
/// us. Held to three waves per SIMD, HLLC spills 140 bytes (48 us). Boundary faces go column by
/// column, their four columns on the cell's four lanes: with all columns on one lane the boundary
/// code, both sides duals, would set the kernel's registers.
template <int FLUX, bool VISC, class VT>
__global__ __launch_bounds__(BLOCK, 2)
void k_jacobian(int ncell, const double* __restrict__ u, const int* __restrict__ nbr,
                const int* __restrict__ face, const FaceGeom* __restrict__ fgeom,
                const double* __restrict__ centre, const int* __restrict__ bcid,
                const GasParams* __restrict__ gpa, const BCTable* __restrict__ bta,
                const BatchArg ba, VT* __restrict__ vals, const double* __restrict__ dt,
                const double* __restrict__ area, double cfl0, double* __restrict__ dtm,
                const int xcd)
{
	// instance: state, matrix, time steps and CFL number are per instance; gpa holds the gas
	// parameters of each instance (one entry for a single solve)
	const long I = ba.list ? ba.list[blockIdx.y] : 0;
	if(I < 0) return;                     // a retired slot of a compacted list
	const GasParams& gp = gpa[I];
	const BCTable& bt = *bta;
	const double cfl = ba.cfl ? ba.cfl[I] : cfl0;
	u += I*4L*ncell;
	vals += I*80L*ncell;
	if(dt) { dt += I*(long)ncell; dtm += I*(long)ncell; }
	// LDS: per side, block entry and (cell, face) the derivatives -- two doubles of padding per
	// entry spread the rows of a block, four entries apart, over the banks --, and the side of
	// the cell's own state (2 boundary: its derivatives are under side 0; 3 none)
	extern __shared__ double lds[];
	const int cpb = jac_cells(blockDim.x), F = 4*cpb, S = F + 2;
	unsigned char* skind = reinterpret_cast<unsigned char*>(lds + 32*S);
	auto sj = [&](int side, int k, int f) -> double& { return lds[(16*side + k)*S + f]; };
	const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
	const bool both = blockDim.x == 64;
	const bool left = both || (wave & 1) == 0, right = both || (wave & 1) == 1;
	const int slot = (both ? 0 : (wave >> 1)*64) + lane;      // 4 cell + face
	const int c0 = xcd_block(xcd)*cpb;
	const int cell = c0 + (slot >> 2), q = slot & 3;
	const int nb = cell < ncell ? nbr[cell*4 + q] : SLOT_UNUSED;
	const bool selfL = nb < 0 || cell < nb;
	if(left) skind[slot] = nb == SLOT_UNUSED ? 3 : nb < 0 ? 2 : selfL ? 0 : 1;
	if(nb >= 0) {
		const FaceGeom G = fgeom[face[cell*4 + q]];
		const double n[2] = { G.nx, G.ny };
		const int cl = selfL ? cell : nb, cr = selfL ? nb : cell;
		double ul[4], ur[4], xl[2] = {0, 0}, xr[2] = {0, 0}, J[16];
		load4(u + 4*cl, ul);
		load4(u + 4*cr, ur);
		if constexpr(VISC) {
			xl[0] = centre[2*cl]; xl[1] = centre[2*cl+1];
			xr[0] = centre[2*cr]; xr[1] = centre[2*cr+1];
		}
		const double sgn = selfL ? G.len : -G.len;
		if(left) {
			side_jacobian<FLUX, VISC, 0>(gp, n, xl, xr, ul, ur, J);
#pragma unroll
			for(int k = 0; k < 16; k++) sj(0, k, slot) = sgn*J[k];
		}
		if(right) {
			side_jacobian<FLUX, VISC, 1>(gp, n, xl, xr, ul, ur, J);
#pragma unroll
			for(int k = 0; k < 16; k++) sj(1, k, slot) = sgn*J[k];
		}
	}
	// boundary faces: the cell's four lanes take a column each; even faces in the left wave, odd
	// ones in the right
	for(int k = 0; k < 4; k++) {
		const int nk = __shfl(nb, (lane & ~3) + k);
		if(nk >= 0 || nk == SLOT_UNUSED || !((k & 1) ? right : left)) continue;
		const FaceGeom G = fgeom[-1 - nk];       // boundary faces are numbered first
		const double n[2] = { G.nx, G.ny };
		double ul[4], xl[2] = {0, 0}, xg[2] = {0, 0}, col[4];
		load4(u + 4*cell, ul);
		if constexpr(VISC) {
			xl[0] = centre[2*cell]; xl[1] = centre[2*cell+1];
			xg[0] = 2.0*G.mx - xl[0]; xg[1] = 2.0*G.my - xl[1];
		}
		boundary_column<FLUX, VISC>(gp, bt, bcid[-1 - nk], n, xl, xg, ul, q, col);
#pragma unroll
		for(int i = 0; i < 4; i++) sj(0, 4*i + q, (slot & ~3) + k) = col[i]*G.len;
	}
	__syncthreads();
	const int nc = min(cpb, ncell - c0);
	// the neighbours' blocks: row r of slot 1 + k
	for(int t = threadIdx.x; t < 16*nc; t += blockDim.x) {
		const int f = t >> 2, r = t & 3, kind = skind[f];
		double row[4];
#pragma unroll
		for(int j = 0; j < 4; j++) {
			const double v = sj(kind == 0 ? 1 : 0, 4*r + j, f);
			row[j] = kind < 2 ? v : 0.0;
		}
		store_row<VT>(vals + (size_t)(c0 + (f >> 2))*80 + 16*(1 + (f & 3)) + 4*r, row);
	}
	// the diagonal block: the own sides of the four faces, in the order (0 + 1) + (2 + 3)
	for(int t = threadIdx.x; t < 4*nc; t += blockDim.x) {
		const int lc = t >> 2, r = t & 3, c = c0 + lc;
		double v[4][4];
#pragma unroll
		for(int k = 0; k < 4; k++) {
			const int kind = skind[4*lc + k];
#pragma unroll
			for(int j = 0; j < 4; j++) {
				const double a = sj(kind == 1 ? 1 : 0, 4*r + j, 4*lc + k);
				v[k][j] = kind == 3 ? 0.0 : a;
			}
		}
		double add = 0.0, row[4];
		if(dt) {
			add = area[c]/(cfl*dt[c]);
			if(r == 0) dtm[c] = add;
		}
#pragma unroll
		for(int j = 0; j < 4; j++)
			row[j] = ((v[0][j] + v[1][j]) + (v[2][j] + v[3][j])) + (j == r ? add : 0.0);
		store_row<VT>(vals + (size_t)c*80 + 4*r, row);
	}
}

template <int FLUX, bool VISC>
static void launch_jac_t(const fvx_disc_s& d, const double* u, void* vals, int prec,
                         const double* dt, double cfl, double* dtm, hipStream_t s,
                         const BatchArg& ba, int nact)
{
	const fvx_mesh_s* m = d.m;
	const int n = m->nelem;
	const int block = d.tune.jac_block, cpb = jac_cells(block);
	const dim3 g((n + cpb - 1)/cpb, nact);
	const size_t lds = 32*(4*(size_t)cpb + 2)*sizeof(double) + 4*(size_t)cpb;
	if(prec == FVX_PREC_F32)
		hipLaunchKernelGGL((k_jacobian<FLUX, VISC, float>), g, dim3(block), lds, s, n, u,
		                   m->d_nbr.p, m->d_face.p, m->d_fgeom.p, m->d_centre.p, d.d_bcid.p,
		                   ba.gp ? ba.gp : d.d_gas.p, d.d_bct.p, ba, static_cast<float*>(vals), dt,
		                   m->d_area.p, cfl, dtm, d.tune.jac_xcd);
	else
		hipLaunchKernelGGL((k_jacobian<FLUX, VISC, double>), g, dim3(block), lds, s, n, u,
		                   m->d_nbr.p, m->d_face.p, m->d_fgeom.p, m->d_centre.p, d.d_bcid.p,
		                   ba.gp ? ba.gp : d.d_gas.p, d.d_bct.p, ba, static_cast<double*>(vals),
		                   dt, m->d_area.p, cfl, dtm, d.tune.jac_xcd);
	FVX_HIP(hipGetLastError());
}

template <int FLUX>
static void launch_jac_v(const fvx_disc_s& d, const double* u, void* vals, int prec,
                         const double* dt, double cfl, double* dtm, hipStream_t s,
                         const BatchArg& ba, int nact)
{
	if(d.pc.viscous) launch_jac_t<FLUX, true>(d, u, vals, prec, dt, cfl, dtm, s, ba, nact);
	else launch_jac_t<FLUX, false>(d, u, vals, prec, dt, cfl, dtm, s, ba, nact);
}

bool jacobian_supported(const fvx_disc_s& d)
{
	const int f = d.nc.conv_numflux_jac;
	if(f != FVX_FLUX_ROE && f != FVX_FLUX_HLLC && f != FVX_FLUX_HLL && f != FVX_FLUX_LLF &&
	   f != FVX_FLUX_AUSM)
		return false;
	for(int i = 0; i < d.pc.nbc; i++) {
		const int k = d.pc.bcs[i].kind;
		if(k == FVX_BC_SUBSONIC_INFLOW || k == FVX_BC_PERIODIC) return false;
	}
	return true;
}

void launch_jacobian(const fvx_disc_s& d, const double* u, void* vals, int prec,
                     const double* dt, double cfl, double* dtm, hipStream_t s,
                     const BatchArg& ba, int nact)
{
	d.prof.start(PROF_JACOBIAN, s);
	switch(d.nc.conv_numflux_jac) {
	case FVX_FLUX_ROE:  launch_jac_v<0>(d, u, vals, prec, dt, cfl, dtm, s, ba, nact); break;
	case FVX_FLUX_HLLC: launch_jac_v<1>(d, u, vals, prec, dt, cfl, dtm, s, ba, nact); break;
	case FVX_FLUX_HLL:  launch_jac_v<2>(d, u, vals, prec, dt, cfl, dtm, s, ba, nact); break;
	case FVX_FLUX_LLF:  launch_jac_v<3>(d, u, vals, prec, dt, cfl, dtm, s, ba, nact); break;
	case FVX_FLUX_AUSM: launch_jac_v<4>(d, u, vals, prec, dt, cfl, dtm, s, ba, nact); break;
	default: throw Error(FVX_ERR_UNSUPPORTED, "flux Jacobian not available for this flux");
	}
	d.prof.stop(s);
}

}
