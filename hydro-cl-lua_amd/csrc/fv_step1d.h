// fv_step1d.h — whole integrator steps of a 1D grid in one launch.
//
// A 1D stage is over in the time a launch takes, and a step of a Runge-Kutta
// integrator is two to four of them. Here a wave takes its cells through all
// stages of a step in registers: a stage's stencil reaches two cells to each side,
// so a wave of 64 cells with a halo of 2 * order on each side outputs
// 64 - 4 * order, and its halo is advanced beside them (the same arithmetic on the
// same states as in the neighbouring wave: the same bits). Between stages, ghost
// lanes take the boundary's values from the lanes of their source cells; a
// periodic ghost's lane is its source cell's twin and advances by itself.
// The stages' states and derivatives stay in registers, so a step reads the state
// once and writes it once, into the other of two buffers (neighbouring waves
// still read this one).
//
// A grid that fits one block (at most STEP1D_WAVES waves) takes many steps per launch: the
// state goes around through LDS, the step's dt is the minimum over the block, and
// nothing leaves the CU in between.
//
// Per step, one launch per stage -> this: Riemann problem of 20011 cells FP32,
// RK2-TVD 11.0 -> 6.4 us (bound by one launch and the latency of two stages; 6.9 with
// the first strip's bookkeeping at the end); Sod on 256 cells FP64 IEEE, forward Euler
// 6.5 -> 3.5 us in one block (the latency of one stage's chain, two barriers and the dt).
#pragma once

#include "fv_stage.h"

namespace hydro {

// waves of a one-block grid at most, so that a lane has 256 registers (enough but for the
// flux-limited GLM-Maxwell FP64 forms, which spill 5 to 27)
constexpr int STEP1D_WAVES = 8;

// output cells of a wave
__host__ __device__ constexpr int step1d_out(int order) { return WAVE - 2 * NG * order; }

// -div F (and the source) of this lane's cell; lanes within two of the wave's
// ends get values of no use (their missing neighbours are stood in for by
// themselves, which keeps the wave on the regular paths)
template <typename R, class E, bool PLM, bool LIM, int FLIM, int SLIM>
__device__ __forceinline__ void derivative_1d(const typename E::Par &par, const StageArgs<R> &a, const GridDesc<R> &g,
	const Cell<R, E> &U, R dt_dx, R *deriv)
{
	using C = Cell<R, E>;
	constexpr int Q = E::Q;
	const int lim = PLM ? 0 : a.limiter;
	C Um, Up;
#pragma unroll
	for (int f = 0; f < C::NV; ++f) {
		Um.v[f] = from_left_or(U.v[f], U.v[f]);
		Up.v[f] = from_right_or(U.v[f], U.v[f]);
	}
	R F[Q];
	if constexpr (PLM) {
		C L, Rr, RL;
		plm_cons<R, E, SLIM, 0>(par, a.limiter, Um, U, Up, L, Rr, dt_dx);
#pragma unroll
		for (int f = 0; f < C::NV; ++f) RL.v[f] = from_left_or(Rr.v[f], Rr.v[f]);
		iface_solve<R, E, 0, ROE_INLINE>(par, RL, L, dt_dx, lim, F);
	} else if constexpr (LIM) {
		Iface<R, E> I;
		iface_prep<R, E, 0>(par, Um, U, I);
		R dWL[E::NW], dWR[E::NW];
#pragma unroll
		for (int k = 0; k < E::NW; ++k) {
			dWL[k] = from_left(I.dW[k]);
			dWR[k] = from_right(I.dW[k]);
		}
		iface_flux<R, E, 0, true, FLIM>(par, I, dWL, dWR, dt_dx, lim, F);
	} else {
		iface_solve<R, E, 0, ROE_INLINE>(par, Um, U, dt_dx, lim, F);
	}
#pragma unroll
	for (int k = 0; k < Q; ++k) {
		const R Fa = flux_on<E>(g, 0) ? F[k] * flux_aov<E, LIM>(g, 0) : R(0);
		deriv[k] = R(0) - (from_right(Fa) - Fa);
		if (!E::FASTM && !g.derivOn) deriv[k] = R(0);
	}
	if constexpr (E::SOURCE) {
		R em[3], ep[3];
		em[0] = Um.v[E::SRC_FIELD];
		ep[0] = Up.v[E::SRC_FIELD];
		E::template source<1>(par, g, U.v, em, ep, deriv);
	}
}

// The boundary's values in the ghost lanes of a stage's new state (integrated
// fields): from the lane of the ghost's source cell, at most 2 * order lanes
// away and inside the part of the wave that is still valid.
template <typename R, class E>
__device__ __forceinline__ void ghost_lanes(const GridDesc<R> &g, const Mapped &m, int x, int lane, Cell<R, E> &U) {
	const int from = min(max(lane + (m.idx - x), 0), WAVE - 1);
	const bool ghost = x < 0 || x >= g.n[0];
#pragma unroll
	for (int f = 0; f < E::Q; ++f) {
		if (!E::active(f)) continue;
		R v = __shfl(U.v[f], from);
		const R fv = g.fixedv[m.fixedFace < 0 ? 0 : m.fixedFace][f];
		if (m.fixedFace >= 0) v = fv;
		else if (m.mirror && E::reflects(f, 0)) v = -v;
		U.v[f] = ghost ? v : U.v[f];
	}
}

template <typename R, template <typename> class EQ, bool PLM, bool LIM, int FLIM, int SLIM>
__global__ void __launch_bounds__(WAVE * STEP1D_WAVES) step1d_kernel(const StepArgs<R> a)
{
	using E = EQ<R>;
	using C = Cell<R, E>;
	constexpr int Q = E::Q;
	extern __shared__ __align__(16) unsigned char step1d_lds[];   // one block: Q planes of n cells
	__shared__ double waveDt[STEP1D_WAVES];
	const GridDesc<R> &g = a.g;
	const typename E::Par par = E::par(a);
	const int lane = threadIdx.x & 63;
	const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int wavesPerBlock = blockDim.x >> 6;
	const bool oneBlock = a.steps > 1;
	const int order = a.order;
	const int n = g.n[0];
	const long item = (long)(a.xcdRemap ? xcd_block(blockIdx.x, a.nBlocks) : (int)blockIdx.x) * wavesPerBlock + w;
	const int out = step1d_out(order), halo = NG * order;
	if (item * out >= n) return;       // whole waves; a grid in one block has no such wave
	const int x = (int)(item * out) - halo + lane;
	const bool outLane = lane >= halo && lane < WAVE - halo && x < n;
	const Mapped m = map_coord(x, n, g.bc[0], g.bc[1], 0);
	Mapped m1;
	m1.idx = 0; m1.mirror = 0; m1.fixedFace = -1;
	// waves with ghosts that are no twins of their source cells
	const bool edge = wave_any((x < 0 && g.bc[0] != HYDRO_BC_PERIODIC) || (x >= n && g.bc[1] != HYDRO_BC_PERIODIC));
	const R *src = g.U[a.src];
	C U;
	load_cell<R, E>(g, src, m, m1, U);
	double dt = stage_dt(a, g);
	double t = 0.;
	if (oneBlock && a.advanceTime) t = g.dev->t;
	if (!oneBlock && item == 0) stage_first_strip(a, g, dt, lane);
	double newDt = INFINITY;           // the block's dt minimum of the last state

	for (int step = 0; step < a.steps; ++step) {
		const R dt_dx = R(dt) / g.dx[0];
		FastestOf<R, E, 1> fw;
		R Us[4][Q], D[3][Q];           // the stages' states and derivatives, in registers: constant indices only
#pragma unroll
		for (int j = 0; j < Q; ++j) {
			Us[0][j] = U.v[j];
			Us[1][j] = Us[2][j] = Us[3][j] = D[0][j] = D[1][j] = D[2][j] = R(0);
		}
#pragma unroll 1
		for (int s = 0; s < order; ++s) {
			R deriv[Q];
			derivative_1d<R, E, PLM, LIM, FLIM, SLIM>(par, a, g, U, dt_dx, deriv);
			// integrator combine (rk.lua:155-174, fe.lua:50), constrainU
			double acc[Q];
#pragma unroll
			for (int j = 0; j < Q; ++j) acc[j] = 0.;
#pragma unroll
			for (int k = 0; k < 4; ++k) {
				if (k > s || a.rkAlpha[s][k] == 0.) continue;
				const double al = a.rkAlpha[s][k];
#pragma unroll
				for (int j = 0; j < Q; ++j)
					if (E::active(j)) acc[j] = acc[j] + (double)Us[k][j] * al;
			}
#pragma unroll
			for (int k = 0; k < 3; ++k) {
				if (k >= s || a.rkBeta[s][k] == 0.) continue;
				const double c = (double)R(a.rkBeta[s][k] * dt);
#pragma unroll
				for (int j = 0; j < Q; ++j)
					if (E::active(j)) acc[j] = acc[j] + (double)D[k][j] * c;
			}
			if (a.rkBeta[s][s] != 0.) {
				const double c = (double)R(a.rkBeta[s][s] * dt);
#pragma unroll
				for (int j = 0; j < Q; ++j)
					if (E::active(j)) acc[j] = acc[j] + (double)deriv[j] * c;
			}
			E::constrain(a.pd, acc);
#pragma unroll
			for (int j = 0; j < Q; ++j) U.v[j] = E::active(j) ? R(acc[j]) : R(0);
			if (s + 1 < order) {
				if (edge) ghost_lanes<R, E>(g, m, x, lane, U);
#pragma unroll
				for (int k = 0; k < 3; ++k) {
					if (k != s) continue;
#pragma unroll
					for (int j = 0; j < Q; ++j) {
						D[k][j] = deriv[j];
						Us[k + 1][j] = U.v[j];
					}
				}
			}
		}
		if (a.reduceSlot >= 0 && outLane) {
			double ud[C::NV], lam[1];
#pragma unroll
			for (int j = 0; j < C::NV; ++j) ud[j] = (double)U.v[j];
			E::template fastest<1>(a.pd, ud, lam);
			fw.add(g.cflScale, lam);
		}
		t = t + dt;
		if (!oneBlock) {
			if (outLane) {
				R *to = a.out >= 0 ? g.U[a.out] : g.ping;
#pragma unroll
				for (int j = 0; j < Q; ++j)
					if (E::active(j)) to[j * g.ps + x] = U.v[j];
			}
			if (a.reduceSlot >= 0) stage_reduce(a, g, fw.dt(g.cflScale), item, lane);
			return;
		}
		// ---- one block: the state around through LDS, the next step's dt
		R *plane = reinterpret_cast<R *>(step1d_lds);
		if (outLane) {
#pragma unroll
			for (int j = 0; j < Q; ++j)
				if (E::active(j)) plane[j * n + x] = U.v[j];
		}
		if (a.reduceSlot >= 0) {
			const double d = wave_min(fw.dt(g.cflScale));
			if (lane == 0) waveDt[w] = d;
		}
		__syncthreads();
		const double dtDone = dt;
		if (a.reduceSlot >= 0) {
			newDt = waveDt[0];
			for (int k = 1; k < wavesPerBlock; ++k) newDt = fmin(newDt, waveDt[k]);
			dt = g.cfl * newDt;
		}
		if (step + 1 < a.steps) {
#pragma unroll
			for (int f = 0; f < Q; ++f) {
				if (!E::active(f)) continue;
				R v = plane[f * n + m.idx];
				const R fv = g.fixedv[m.fixedFace < 0 ? 0 : m.fixedFace][f];
				if (m.fixedFace >= 0) v = fv;
				else if (m.mirror && E::reflects(f, 0)) v = -v;
				U.v[f] = v;
			}
			__syncthreads();           // read by every wave before the next step writes it
		} else {
			R *to = g.U[0];
			if (outLane) {
#pragma unroll
				for (int j = 0; j < Q; ++j)
					if (E::active(j)) to[j * g.ps + x] = U.v[j];
			}
			if (w == 0) {
				if (a.reduceSlot >= 0) {
					// the slots as the last of these steps leaves them
#pragma unroll
					for (int k = 0; k < 3; ++k)
						g.dev->dtmin[k][lane] = k == a.reduceSlot && lane == 0 ? newDt : (double)INFINITY;
				}
				if (a.advanceTime && lane == 0) {
					g.dev->t = t;
					g.dev->dt = dtDone;
				}
			}
		}
	}
}

} // namespace hydro
