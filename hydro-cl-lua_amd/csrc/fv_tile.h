// fv_tile.h — the fused 2D stage kernel for grids that do not fill the device:
// a tile of rows, one row per wave.
//
// The same stage as stage_kernel (fv_stage.h), cut the other way. There a wave
// marches several rows of a strip, which shares the work of neighbouring rows
// but takes as long as those rows one after the other; on a grid of up to some
// 500^2 cells every wave of the launch is resident at once, one or two per SIMD,
// and the launch lasts one wave's march (13-16 us from 64^2 to 512^2, FP64 and
// FP32 alike). Here a block of TILE_W row waves and one halo wave owns 64
// columns (60 with a flux limiter or a source term) of TILE_W rows:
//   row wave w loads rows y-2 .. y+1 of its column, computes the interface below
//     its row (y) and the one left of its cells (x), and takes the flux above its
//     row from the next wave through LDS;
//   the halo wave computes the block's top interface, and the strip's edge
//     interfaces of the block's rows (the row waves' lanes 0 and 63 load the
//     cells beside the strip themselves).
// Every wave has two interfaces to compute, and the block one barrier (two with
// a flux limiter, which exchanges the characteristic jumps first). Both Roe
// forms fit (98 VGPRs FP64), so no wave leaves its row to another form.
// One row per wave costs a launch per row of work, and the top interface of
// every three rows twice: beyond the sizes of tile_form (fv_host.h) the marching
// kernel is the faster one. Per stage, marching -> tile: KH 64^2 FP64 13.6 -> 6.4,
// 256^2 13.7 -> 7.8, 400^2 13.9 -> 11.5, 512^2 14.8 -> 15.0 us; 256^2 FP32 11.8 ->
// 6.9, flux-limited FP64 15.7 -> 8.7, IEEE 29.8 -> 12.9, GLM-Maxwell FP32 11.8 ->
// 7.3, shallow water 13.2 -> 7.9 us. Blocks of 7 row waves: 7.5 us at 64^2, 16.3
// at 512^2 (more of a block's time is its slowest wave's).
#pragma once

#include "fv_stage.h"

namespace hydro {

constexpr int TILE_SIDE = 4;           // slots per side of the strip-edge fluxes
static_assert(TILE_W <= TILE_SIDE, "a slot per row");

// reconstructions that take dt need it before the interfaces; the others only
// for the combine, so that its load is waited for behind the stencil's
template <class E>
__host__ __device__ constexpr bool tile_late_dt(bool lim) {
	return !lim && !E::PLM_EIG && !E::PLM_CONS_FLUX && !E::PLM_EIG_PRIM && !E::PLM_EIG_PRIM_REF;
}

template <typename R, class E, bool LIM, bool EDGES>
struct TileLds {
	R f[TILE_W + 1][E::Q][WAVE];                           // slot w: flux of the interface below row w
	R d[LIM ? TILE_W + 2 : 1][LIM ? E::NW : 1][WAVE];      // slot k: dW of the interface below row k - 1
	R ef[EDGES ? E::Q : 1][EDGES ? 2 * TILE_SIDE : 1];     // strip-edge fluxes: left of row w at w, right at TILE_SIDE + w
};

template <typename R, template <typename> class EQ, bool PLM, bool LIM, int FLIM, int SLIM>
__global__ void __launch_bounds__(WAVE * TILE_WAVES) stage_kernel_tile(const StageArgs<R> a)
{
	using E = EQ<R>;
	using C = Cell<R, E>;
	constexpr int Q = E::Q, W = TILE_W;
	constexpr bool EDGES = tile_edges(E::SOURCE, LIM);
	__shared__ TileLds<R, E, LIM, EDGES> sh;
	const int lane = threadIdx.x & 63;
	const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int blk = a.xcdRemap ? xcd_block(blockIdx.x, a.nBlocks) : (int)blockIdx.x;
	const GridDesc<R> &g = a.g;
	const typename E::Par par = E::par(a);
	const int lim = PLM ? 0 : a.limiter;
	const int slim = a.limiter;
	const int nx = g.n[0], ny = g.n[1];
	const int sx = blk % g.stripsX, by = blk / g.stripsX;
	const R *src = g.U[a.src];
	const int x = EDGES ? sx * STRIP_OUT + lane : sx * strip_out(false) - NG + lane;
	const int y0 = by * W, y = y0 + w;
	const Mapped mx = map_coord(x, nx, g.bc[0], g.bc[1], 0);
	const bool xPlain = wave_all(mx.fixedFace < 0 && !mx.mirror);
	auto loadRow = [&](int r, C &c) {
		Mapped my = map_coord(r, ny, g.bc[2], g.bc[3], 2);
		if (xPlain && my.fixedFace < 0 && !my.mirror) load_plain<R, E>(g, src, (long)my.idx * g.step1 + mx.idx, c);
		else load_cell<R, E>(g, src, mx, my, c);
	};
	C c1, c2, c3;      // rows y-1, y, y+1
	const double dtRaw = a.dtSlot >= 0 ? g.dev->dtmin[a.dtSlot][lane] : 0.;
	double dt = 0.;
	R dt_dx0 = R(0), dt_dx1 = R(0);
	constexpr bool EARLY_DT = !tile_late_dt<E>(LIM);
	auto get_dt = [&]() {
		dt = a.dtSlot >= 0 ? g.cfl * wave_min(dtRaw) : a.hostDt;
		dt_dx0 = R(dt) / g.dx[0];
		dt_dx1 = R(dt) / g.dx[1];
	};
	FastestOf<R, E, 2> fw;

	// ---- y: the flux of the interface below row y
	R FaY[Q];
	{
		R F[Q];
		loadRow(y - 1, c1);
		loadRow(y, c2);
		if constexpr (PLM) {
			C c0, L1, R1, L2, R2;
			loadRow(y - 2, c0);
			loadRow(y + 1, c3);
			if constexpr (EARLY_DT) get_dt();
			plm_cons<R, E, SLIM, 1>(par, slim, c0, c1, c2, L1, R1, dt_dx1);
			plm_cons<R, E, SLIM, 1>(par, slim, c1, c2, c3, L2, R2, dt_dx1);
			iface_solve<R, E, 1, ROE_INLINE>(par, R1, L2, dt_dx1, lim, F);
		} else if constexpr (LIM) {
			get_dt();
			Iface<R, E> I;
			R dWL[E::NW], dWR[E::NW];
			iface_prep<R, E, 1>(par, c1, c2, I);
#pragma unroll
			for (int j = 0; j < E::NW; ++j) sh.d[w + 1][j][lane] = I.dW[j];
			if (w == W) {
				// the jumps next to the block's first and last interfaces
				C c0;
				Iface<R, E> Ie;
				loadRow(y + 1, c3);
				iface_prep<R, E, 1>(par, c2, c3, Ie);     // y0+W+1/2: for its own flux
#pragma unroll
				for (int j = 0; j < E::NW; ++j) dWR[j] = Ie.dW[j];
				loadRow(y0 - 2, c0);
				loadRow(y0 - 1, c1);
				iface_prep<R, E, 1>(par, c0, c1, Ie);     // y0-3/2
#pragma unroll
				for (int j = 0; j < E::NW; ++j) sh.d[0][j][lane] = Ie.dW[j];
			} else if constexpr (E::SOURCE) {
				loadRow(y + 1, c3);
			}
			__syncthreads();
#pragma unroll
			for (int j = 0; j < E::NW; ++j) {
				dWL[j] = sh.d[w][j][lane];
				if (w < W) dWR[j] = sh.d[w + 2][j][lane];
			}
			iface_flux<R, E, 1, true, FLIM>(par, I, dWL, dWR, dt_dx1, lim, F);
		} else {
			if constexpr (E::SOURCE) loadRow(y + 1, c3);
			iface_solve<R, E, 1, ROE_INLINE>(par, c1, c2, dt_dx1, lim, F);
		}
#pragma unroll
		for (int j = 0; j < Q; ++j) {
			FaY[j] = flux_on<E>(g, 1) ? F[j] * flux_aov<E, LIM>(g, 1) : R(0);
			if (E::active(j)) sh.f[w][j][lane] = FaY[j];
		}
	}

	if (w == W) {
		// ---- the halo wave: the strip's edge interfaces of the block's rows
		if constexpr (EDGES) {
			const int j = lane & (TILE_SIDE - 1);
			const bool right = (lane & TILE_SIDE) != 0;
			const int xb = sx * STRIP_OUT + (right ? STRIP_OUT : 0);
			const Mapped myb = map_coord(y0 + (j < W ? j : 0), ny, g.bc[2], g.bc[3], 2);
			C cb[4];
			Mapped mxb[4];
			bool plain = myb.fixedFace < 0 && !myb.mirror;
#pragma unroll
			for (int k = 0; k < 4; ++k) {
				mxb[k] = map_coord(xb - 2 + k, nx, g.bc[0], g.bc[1], 0);
				plain = plain && mxb[k].fixedFace < 0 && !mxb[k].mirror;
			}
			if (wave_all(plain)) {
#pragma unroll
				for (int k = 0; k < 4; ++k) load_plain<R, E>(g, src, (long)myb.idx * g.step1 + mxb[k].idx, cb[k]);
			} else {
#pragma unroll
				for (int k = 0; k < 4; ++k) load_cell<R, E>(g, src, mxb[k], myb, cb[k]);
			}
			R Fa[Q], dW[E::NW];
			bool ok;
			edge_flux<R, E, PLM, LIM, FLIM, SLIM, ROE_INLINE>(par, lim, slim, cb, dt_dx0, flux_on<E>(g, 0), flux_aov<E, LIM>(g, 0),
				Fa, dW, ok);
			if (lane < 2 * TILE_SIDE) {
#pragma unroll
				for (int q = 0; q < Q; ++q) sh.ef[q][lane] = Fa[q];
			}
		}
		__syncthreads();
		return;
	}

	// ---- x on row y (lanes)
	C Um, Up;
	if constexpr (EDGES && PLM) {
		// the cells beside the strip, for lanes 0 and 63
		C ce = c2;
		if (lane == 0 || lane == WAVE - 1) {
			const Mapped me = map_coord(lane == 0 ? x - 1 : x + 1, nx, g.bc[0], g.bc[1], 0);
			const Mapped my = map_coord(y, ny, g.bc[2], g.bc[3], 2);
			load_cell<R, E>(g, src, me, my, ce);
		}
#pragma unroll
		for (int f = 0; f < C::NV; ++f) {
			Um.v[f] = from_left_or(c2.v[f], ce.v[f]);
			Up.v[f] = from_right_or(c2.v[f], ce.v[f]);
		}
	} else {
#pragma unroll
		for (int f = 0; f < C::NV; ++f) {
			Um.v[f] = from_left_or(c2.v[f], c2.v[f]);
			Up.v[f] = from_right_or(c2.v[f], c2.v[f]);
		}
	}
	R Fx[Q], divx[Q];
	if constexpr (PLM) {
		C Lx, Rx, RxL;
		plm_cons<R, E, SLIM, 0>(par, slim, Um, c2, Up, Lx, Rx, dt_dx0);
#pragma unroll
		for (int f = 0; f < C::NV; ++f) RxL.v[f] = from_left_or(Rx.v[f], Rx.v[f]);
		iface_solve<R, E, 0, ROE_INLINE>(par, RxL, Lx, dt_dx0, lim, Fx);
	} else if constexpr (LIM) {
		Iface<R, E> I;
		iface_prep<R, E, 0>(par, Um, c2, I);
		R dWL[E::NW], dWR[E::NW];
#pragma unroll
		for (int k = 0; k < E::NW; ++k) {
			dWL[k] = from_left(I.dW[k]);
			dWR[k] = from_right(I.dW[k]);
		}
		iface_flux<R, E, 0, true, FLIM>(par, I, dWL, dWR, dt_dx0, lim, Fx);
	} else {
		iface_solve<R, E, 0, ROE_INLINE>(par, Um, c2, dt_dx0, lim, Fx);
	}
	if constexpr (!EARLY_DT) get_dt();
	if (blk == 0 && w == 0) stage_first_strip(a, g, dt, lane);
	__syncthreads();
#pragma unroll
	for (int k = 0; k < Q; ++k) {
		R Fa = flux_on<E>(g, 0) ? Fx[k] * flux_aov<E, LIM>(g, 0) : R(0);
		R FaR;
		if constexpr (EDGES) {
			const R e = sh.ef[k][lane == WAVE - 1 ? TILE_SIDE + w : w];
			Fa = lane == 0 ? e : Fa;
			FaR = from_right_or(Fa, e);
		} else {
			FaR = from_right(Fa);
		}
		divx[k] = R(0) - (FaR - Fa);
	}
	R deriv[Q];
#pragma unroll
	for (int j = 0; j < Q; ++j) {
		const R dyterm = E::active(j) ? sh.f[w + 1][j][lane] - FaY[j] : R(0);
		deriv[j] = divx[j] - dyterm;
		if (!E::FASTM && !g.derivOn) deriv[j] = R(0);
	}
	if constexpr (E::SOURCE) {
		R em[3], ep[3];
		constexpr int SF = E::SRC_FIELD;
		em[0] = Um.v[SF]; ep[0] = Up.v[SF];
		em[1] = c1.v[SF]; ep[1] = c3.v[SF];
		E::template source<2>(par, g, c2.v, em, ep, deriv);
	}
	const bool outLane = (EDGES ? x < nx : lane >= NG && lane < WAVE - NG && x < nx) && y < ny;
	if (outLane) {
		R *out = a.out >= 0 ? g.U[a.out] : g.ping;
		R *storeD = a.storeD >= 0 ? g.D[a.storeD] : nullptr;
		finish_cell<R, E, 2>(a, g, (long)y * g.step1 + x, c2, deriv, dt, out, storeD, fw);
	}
	if (a.reduceSlot >= 0) stage_reduce(a, g, fw.dt(g.cflScale), (long)blk * W + w, lane);
}

} // namespace hydro
