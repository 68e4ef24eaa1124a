// fv_common.h — device-side building blocks shared by every stage kernel:
// the kernel argument block, boundary-mapped loads of the structure-of-arrays
// state, and 64-lane DPP neighbour exchange.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/hydro_hip.h"
#include "fv_math.h"

namespace hydro {

constexpr int NG = 2;              // numGhost (gridsolver.lua:41)
constexpr int WAVE = 64;           // CDNA wavefront
// Flux id of the kernels of the Roe flux with Harten's entropy fix
// (roe.cl:83-106); a template choice of its own, so that the kernels without
// the fix carry no test for it.
constexpr int FLUX_ROE_ENTROPY_FIX = 16;
constexpr int STRIP_OUT = WAVE;    // output columns per wave strip with edge passes
// Strips whose edge interfaces come from an edge pass output 64 columns; the
// others load a 2-cell halo in lanes 0-1 and 62-63 and output 60: 1D strips
// (a single row, too short to repay the pass) and equations with a source
// term, which reads the x neighbours' static fields (GLM-Maxwell: 12 state
// reals per cell make the pass's gathers cost more than the halo lanes,
// measured; shallow water: the depth).
__host__ __device__ constexpr int strip_out(bool edges) { return edges ? STRIP_OUT : WAVE - 2 * NG; }
__host__ __device__ constexpr bool strip_edges(int dim, bool source) { return dim >= 2 && !source; }
constexpr int EDGE_ROWS = WAVE / 2;// rows per wave item at most (2D): the strip-edge
                                   // interfaces of each row take a lane per side
constexpr int EDGE_PLANES = 16;    // planes per block chunk at most (3D)

// 2D tile kernel (fv_tile.h): a block is TILE_W row waves, a row each, and one
// halo wave. Its strips have 64 columns, with edge interfaces from the halo wave;
// with a flux limiter an edge takes three interface preparations, twice a row's:
// there, as with a source term, the strip loads a halo and outputs 60.
constexpr int TILE_W = 3;
constexpr int TILE_WAVES = TILE_W + 1;
__host__ __device__ constexpr bool tile_edges(bool source, bool lim) { return !source && !lim; }

// 3D stage kernel: a block is W row waves (rows of a strip that share one
// plane through LDS) and one halo wave that loads the rows outside the block
// and computes the y interfaces no row owns, so that the row waves do equal
// work between barriers. Four waves, so that several blocks fit per CU and
// one block's barrier waits are covered by the others' work. MIN_BLOCKS
// bounds the registers (FP32: four blocks per CU, 128 VGPRs: the flux-limited
// superbee and 'plm athena' kernels, at 132 on their own, 256 and 435 us against 205
// and 359 at 200x180x160, with 5 registers spilled, as five other FP32 kernels have; FP64 takes what it needs: capped, its kernels spill).
template <typename R>
struct Block3 {
	static constexpr int W = 3;
	static constexpr int WAVES = W + 1;
	static constexpr int MIN_BLOCKS = sizeof(R) == 4 ? 4 : 1;
};

// Device-resident per-solver scalars: dt minima rotate through three slots so
// a step can read one, reduce into the next and clear the third.
constexpr int DT_LANES = 64;       // dt minima are spread over 64 addresses
struct DevScalars {
	double dtmin[3][DT_LANES];
	double t;
	double dt;
	unsigned nonFinite;       // set by nonfinite_kernel
	unsigned pad0[2];
	unsigned ticket;          // blocks of a statistics pass that have finished, 0 between launches
	double pad[4];
};

// Boundary description of one axis, resolved on the host.
struct AxisBC {
	int n;            // interior cells
	int kind[2];      // HYDRO_BC_* at min / max
};

// Cell lengths as the CFL step takes them (FastestWave)
struct CflScale {
	double dx[3];      // cell lengths
	double len;        // the first positive one, INFINITY if there is none
	double scale[3];   // len / dx, 0 for an axis that counts for nothing
};

// Everything that is specific to one grid: its buffers, shape, boundaries,
// metric factors, launch decomposition and device scalars. The plain solver
// passes one by value; a batch keeps an array of them in device memory.
template <typename R>
struct GridDesc {
	R *U[4];                  // stage states U^(0..order-1); U[0] holds the solver state
	R *D[4];                  // stored stage derivatives (tables whose later rows use them)
	R *ping;                  // forward-Euler output (swapped with U[0] after a step)
	const R *stat;            // static (non-integrated) planes: GLM-Maxwell, shallow water
	int n[3];                 // interior cells
	long ps;                  // plane stride (reals)
	long step1;               // row stride (= n[0])
	int bc[6];                // HYDRO_BC_* per face
	R fixedv[6][HYDRO_MAX_STATES];   // HYDRO_BC_FIXED ghost values
	R areaOverVol[3];         // areaL * (1 / volume) per side (fvsolver.cl:64-102)
	int derivOn;              // volume > 1e-7 (fvsolver.cl:97)
	int fluxOn[3];            // cell_area > 1e-7 (fvsolver.lua:105)
	R aovFast[3];             // FAST kernels: areaOverVol where flux and derivative are on, else 0
	R aovHalf[3];             // half of it, for the Roe form that returns twice the flux
	R dx[3];
	R invdx[3];               // 1 / dx in the stored precision (glm-maxwell.cl:351)
	R inv2dx[3];              // 1 / (2 dx) in the stored precision (makepartial.lua:105-108)
	CflScale cflScale;
	double cfl;
	int stripsX, stripsY, rowsPerWave;   // 3D: stripsY counts blocks of Block3::W rows, rowsPerWave planes per chunk
	int active;               // batch: grid takes part in the launch
	long itemBase;            // batch: first work item (wave strip) of this grid
	long nItems;              // stripsX * stripsY
	DevScalars *dev;          // dt slots and time of this grid
	int stepsLeft;            // batch: steps still to run in the current tick
	int stripsZ;              // 3D: plane chunks of rowsPerWave planes
};

// Equation parameters in double: constrainU and the per-cell dt run in double
// in every stored precision.
struct EqnParD {
	double gamma, rhoMin, PMin;   // Euler (euler.lua:192-197)
	double eIntSafe;              // Euler: E - EKin from which on P is clear of PMin, 2 PMin / (gamma - 1) or more
	double divPhi, divPsi;        // GLM-Maxwell (glm-maxwell.lua:110-111)
	double gravity;               // shallow water (shallow-water.lua:167)
};

// Uniform for one launch: the stage's row of the Shu-Osher table (as buffer
// indices), the dt protocol and the equation parameters.
template <typename R>
struct StageArgs {
	int src;                  // buffer index of the stage whose derivative is taken
	int out;                  // output buffer index, -1: ping
	int accU[4];              // alpha terms, reference order
	double alpha[4];
	int nAlpha;
	int accD[3];              // stored derivatives of earlier stages (beta terms)
	double beta[3];
	int nStoredD;
	int storeD;               // store this stage's derivative into D[storeD] (-1: no)
	double betaNew;           // beta of this stage's derivative (0: not used)
	// dt: device slot (cfl * dtmin[slot]) or a host value
	int dtSlot;               // -1: use hostDt
	double hostDt;
	int resetSlot;            // slot to clear to +inf, -1 none
	int reduceSlot;           // slot to min-reduce the new state's dt into, -1 none
	int advanceTime;          // t += dt, dt stored
	int steps;                // whole steps of the launch (then these are a StepArgs's), 0: a stage
	int tile;                 // plain 2D launch of the tile kernel (fv_tile.h)
	int shareEdges;           // plain 2D launch: one strip-edge pass per block of 4 x-adjacent strips
	int stepInTick;           // batch: skip grids with stepsLeft <= stepInTick
	// equation parameters in the stencil type and in double (for the FP64
	// accumulation, constrainU and dt work of the FP32 form)
	R gamma, rhoMin, PMin, divPhi, divPsi, gravity;
	R roeFixFactor;           // Roe, Euler: Harten's entropy fix factor (roe.cl:83-106)
	EqnParD pd;
	int limiter;              // flux or slope limiter index (runtime switch form)
	int xcdRemap;
	int nBlocks;
	// one grid (plain launch) or a batch (persistent launch)
	GridDesc<R> g;
	const GridDesc<R> *grids;
	int nGrids;
	long totalItems;
};

// Of a launch of whole 1D steps (step1d_kernel): all stages' rows of the table too. Not
// in StageArgs: with these 256 bytes in every launch's arguments a 1D stage took
// .4 us longer (FP32, 1000 cells).
template <typename R>
struct StepArgs : StageArgs<R> {
	double rkAlpha[4][4], rkBeta[4][4];
	int order;
};

// ---------------------------------------------------------------- lane moves
// Lane l receives lane l-1's value (wave_shr:1) / lane l+1's (wave_shl:1);
// the lane without a source (0 / 63) receives 0 (bound_ctrl: no old value to
// set up first). With zero fill, FP32 users of a shifted value take the shift
// as a DPP operand (no move).
__device__ __forceinline__ int dpp_from_left_i(int v) {
	return __builtin_amdgcn_update_dpp(0, v, 0x138, 0xF, 0xF, true);
}
__device__ __forceinline__ int dpp_from_right_i(int v) {
	return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xF, 0xF, true);
}
__device__ __forceinline__ double from_left(double v) {
	int2 p = __builtin_bit_cast(int2, v);
	p.x = dpp_from_left_i(p.x);
	p.y = dpp_from_left_i(p.y);
	return __builtin_bit_cast(double, p);
}
__device__ __forceinline__ double from_right(double v) {
	int2 p = __builtin_bit_cast(int2, v);
	p.x = dpp_from_right_i(p.x);
	p.y = dpp_from_right_i(p.y);
	return __builtin_bit_cast(double, p);
}
__device__ __forceinline__ float from_left(float v) {
	return __builtin_bit_cast(float, dpp_from_left_i(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float from_right(float v) {
	return __builtin_bit_cast(float, dpp_from_right_i(__builtin_bit_cast(int, v)));
}

// The same shifts with the empty lane (0 / 63) taking `edge` instead of 0:
// the DPP move's old operand, so no select is needed.
__device__ __forceinline__ double from_left_or(double v, double edge) {
	int2 p = __builtin_bit_cast(int2, v), e = __builtin_bit_cast(int2, edge);
	p.x = __builtin_amdgcn_update_dpp(e.x, p.x, 0x138, 0xF, 0xF, false);
	p.y = __builtin_amdgcn_update_dpp(e.y, p.y, 0x138, 0xF, 0xF, false);
	return __builtin_bit_cast(double, p);
}
__device__ __forceinline__ double from_right_or(double v, double edge) {
	int2 p = __builtin_bit_cast(int2, v), e = __builtin_bit_cast(int2, edge);
	p.x = __builtin_amdgcn_update_dpp(e.x, p.x, 0x130, 0xF, 0xF, false);
	p.y = __builtin_amdgcn_update_dpp(e.y, p.y, 0x130, 0xF, 0xF, false);
	return __builtin_bit_cast(double, p);
}
__device__ __forceinline__ float from_left_or(float v, float edge) {
	return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge),
		__builtin_bit_cast(int, v), 0x138, 0xF, 0xF, false));
}
__device__ __forceinline__ float from_right_or(float v, float edge) {
	return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, edge),
		__builtin_bit_cast(int, v), 0x130, 0xF, 0xF, false));
}

// ------------------------------------------------------- boundary mapping
// A ghost coordinate maps to an interior source cell, a sign for mirror
// reflection, or a fixed value (gridsolver.lua:630-780). The reference fills
// ghosts axis by axis (x, then y, then z), so a later axis wins at corners:
// callers resolve z first, then y, then x.
struct Mapped {
	int idx;      // interior coordinate
	int mirror;   // 1 if the normal vector component flips
	int fixedFace;// face index when a fixed value applies, else -1
};

__device__ __forceinline__ Mapped map_coord(int c, int n, int kmin, int kmax, int faceMin) {
	Mapped m;
	m.idx = c;
	m.mirror = 0;
	m.fixedFace = -1;
	if (c < 0) {
		switch (kmin) {
		case HYDRO_BC_PERIODIC: m.idx = ((c % n) + n) % n; break;
		case HYDRO_BC_MIRROR: m.idx = -1 - c; m.mirror = 1; break;
		case HYDRO_BC_FREEFLOW: m.idx = 0; break;
		default: m.idx = 0; m.fixedFace = faceMin; break;
		}
	} else if (c >= n) {
		switch (kmax) {
		case HYDRO_BC_PERIODIC: m.idx = c % n; break;
		case HYDRO_BC_MIRROR: m.idx = 2 * n - 1 - c; m.mirror = 1; break;
		case HYDRO_BC_FREEFLOW: m.idx = n - 1; break;
		default: m.idx = n - 1; m.fixedFace = faceMin + 1; break;
		}
	}
	// guard tiny grids (n < ghost width): keep every access in bounds
	if (m.idx < 0) m.idx = 0;
	if (m.idx >= n) m.idx = n - 1;
	return m;
}

// Minimum over the wave's 64 lanes, in every lane: four DPP row shifts and the
// two row broadcasts bring it to lane 63 (a lane without a source keeps its own
// value), a pair of readlanes spreads it. Every stage kernel starts by taking
// its dt this way, alone on its latency: against six dependent ds_bpermute
// pairs a launch is .3-.5 us shorter at every grid size.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_min_step(double v) {
	const int2 p = __builtin_bit_cast(int2, v);
	int2 q;
	q.x = __builtin_amdgcn_update_dpp(p.x, p.x, CTRL, ROWS, 0xF, false);
	q.y = __builtin_amdgcn_update_dpp(p.y, p.y, CTRL, ROWS, 0xF, false);
	const double o = __builtin_bit_cast(double, q);
	return o < v ? o : v;
}
__device__ __forceinline__ double wave_min(double v) {
	v = dpp_min_step<0x111, 0xF>(v);     // row_shr:1
	v = dpp_min_step<0x112, 0xF>(v);     // row_shr:2
	v = dpp_min_step<0x114, 0xF>(v);     // row_shr:4
	v = dpp_min_step<0x118, 0xF>(v);     // row_shr:8: lane 15 of each row
	v = dpp_min_step<0x142, 0xA>(v);     // row_bcast:15 into rows 1 and 3
	v = dpp_min_step<0x143, 0xC>(v);     // row_bcast:31 into rows 2 and 3
	int2 p = __builtin_bit_cast(int2, v);
	p.x = __builtin_amdgcn_readlane(p.x, 63);
	p.y = __builtin_amdgcn_readlane(p.y, 63);
	return __builtin_bit_cast(double, p);
}

// min over the 64 sub-slots of a dt slot: one coalesced load per wave
__device__ __forceinline__ double read_dt_slot(const DevScalars *d, int slot) {
	double v = d->dtmin[slot][threadIdx.x & 63];
	return wave_min(v);
}

__device__ __forceinline__ void atomic_min_pos(double *p, double v) {
	// positive doubles (and +inf) order like their bit patterns
	atomicMin(reinterpret_cast<unsigned long long *>(p), (unsigned long long)__double_as_longlong(v));
}

// The CFL step of the cells a lane has seen (calcDT.cl:38-73: the minimum of
// dx / max(1e-9, |lambda|) over cells and axes) from the fastest wave of each
// axis: division is monotonic, so dx / max is the minimum, with one division per
// axis and wave in place of one per axis and cell. ONE (the FP64 FAST kernels):
// one value, every axis' waves scaled to the first axis' cell length (an exact 1
// where the lengths are equal), two registers less through the row loop.
template <int DIM, bool FAST, bool ONE>
struct FastestWave {
	static constexpr int N = ONE ? 1 : DIM;
	double lam[N];
	bool seen;
	__device__ __forceinline__ FastestWave() : seen(false) {
#pragma unroll
		for (int s = 0; s < N; ++s) lam[s] = 0.;
	}
	// l: a cell's fastest wave per axis
	__device__ __forceinline__ void add(const CflScale &c, const double *l) {
#pragma unroll
		for (int s = 0; s < DIM; ++s) {
			if constexpr (ONE) lam[0] = fmax(lam[0], fmax(1e-9, l[s]) * c.scale[s]);
			else lam[s] = fmax(lam[s], l[s]);
		}
		seen = true;
	}
	__device__ __forceinline__ double dt(const CflScale &c) const {
		using MD = Math<double, FAST>;
		double d = INFINITY;
		if constexpr (ONE) {
			d = MD::div(c.len, lam[0]);
		} else {
#pragma unroll
			for (int s = 0; s < DIM; ++s)
				if (c.dx[s] > 0.) d = fmin(d, MD::div(c.dx[s], fmax(1e-9, lam[s])));
		}
		return seen ? d : INFINITY;
	}
};
template <typename R, class E, int DIM>
using FastestOf = FastestWave<DIM, E::FASTM, E::FASTM && sizeof(R) == 8>;

// Logical block id with blocks spread so that each XCD (blocks are dealt
// round-robin over the 8 XCDs) gets a contiguous range of logical ids, so
// neighbouring strips share an L2. A bijection for any block count.
__device__ __forceinline__ int xcd_block(int b, int nBlocks) {
	int q = nBlocks >> 3, r = nBlocks & 7;
	int x = b & 7;
	int start = x * q + (x < r ? x : r);
	return start + (b >> 3);
}

} // namespace hydro
