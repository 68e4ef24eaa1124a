// fv_host.h — host-side internals shared by the C ABI translation units:
// error reporting, Shu-Osher tables, the Grid record (one solver's device
// state), its layout conversion to and from the reference's ghosted cons_t
// buffers, and the argument blocks of the stage kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <string>
#include <thread>
#include <vector>

#include "../../include/hydro_hip.h"
#include "fv_common.h"
#include "fv_launch.h"
#include "fv_aux.h"

namespace hydro {

// ------------------------------------------------------------------ errors
std::string &hydro_err_buf();   // thread-local last error (hydro_hip.cpp)

static inline int fail(const char *fmt, ...) {
	char buf[1024];
	va_list ap;
	va_start(ap, fmt);
	vsnprintf(buf, sizeof buf, fmt, ap);
	va_end(ap);
	hydro_err_buf() = buf;
	return -1;
}

#define HIPCHECK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) \
	return fail("%s failed: %s (%s:%d)", #x, hipGetErrorString(e_), __FILE__, __LINE__); } while (0)

static inline void ignore(hipError_t) {}

static inline int num_states(int eqn) {
	return eqn == HYDRO_EQN_EULER ? 6 : eqn == HYDRO_EQN_GLM_MAXWELL ? 12 : eqn == HYDRO_EQN_SHALLOW_WATER ? 5 : -1;
}
static inline int num_int_states(int eqn) {
	return eqn == HYDRO_EQN_EULER ? 5 : eqn == HYDRO_EQN_GLM_MAXWELL ? 8 : eqn == HYDRO_EQN_SHALLOW_WATER ? 4 : -1;
}
// static (non-integrated) planes on the device: GLM-Maxwell's rhoCharge,
// sigma, sqrt_1_eps, sqrt_1_mu; the shallow water depth (Euler's ePot stays on
// the host)
static inline int num_static_states(int eqn) {
	return eqn == HYDRO_EQN_GLM_MAXWELL ? 4 : eqn == HYDRO_EQN_SHALLOW_WATER ? 1 : 0;
}
// equations with an addSource step, whose strips load a halo instead of
// taking an edge pass (the source reads the x neighbours' static fields)
static inline bool eqn_has_source(int eqn) { return eqn == HYDRO_EQN_GLM_MAXWELL || eqn == HYDRO_EQN_SHALLOW_WATER; }

static inline EqnParD eqn_par_d(const hydro_cfg &c) {
	EqnParD p;
	p.gamma = c.gamma;
	p.rhoMin = c.rho_min;
	p.PMin = c.P_min;
	// (a P above 0 is above a PMin below it; where P falls with the energy or the density
	// may be negative, none is safe: nothing compares above a NaN)
	p.eIntSafe = c.gamma > 1 && c.rho_min >= 0 ? std::max(0., 2. * c.P_min / (c.gamma - 1.)) : NAN;
	p.divPhi = c.div_phi_wavespeed;
	p.divPsi = c.div_psi_wavespeed;
	p.gravity = c.gravity;
	return p;
}

static inline void cfg_default(hydro_cfg *c) {
	std::memset(c, 0, sizeof *c);
	c->dim = 1;
	for (int i = 0; i < 3; ++i) {
		c->size[i] = 1;
		c->mins[i] = -1;
		c->maxs[i] = 1;
	}
	c->eqn = HYDRO_EQN_EULER;
	c->flux = HYDRO_FLUX_ROE;
	c->flux_limiter = HYDRO_LIMITER_DONOR_CELL;
	c->plm = HYDRO_PLM_NONE;
	c->slope_limiter = HYDRO_LIMITER_DONOR_CELL;
	c->integrator = HYDRO_INT_FORWARD_EULER;
	c->cfl = .5;
	c->roe_entropy_fix_factor = .2;
	c->gravity = 1;
	for (int i = 0; i < 6; ++i) c->boundary[i] = HYDRO_BC_FREEFLOW;
	c->precision = HYDRO_REAL_F64;
	c->gamma = 7. / 5.;
	c->rho_min = 1e-7;
	c->P_min = 1e-7;
	c->div_phi_wavespeed = 1;
	c->div_psi_wavespeed = 1;
}

// --------------------------------------------------------- Shu-Osher tables
// hydro/int/all.lua:10-160 (rows = stages, columns = k); forward Euler is a
// one-stage table here (fe.lua:33-49 computes U + dt L(U) as well).
struct RKTable {
	int order;
	double a[4][4], b[4][4];
};

static bool rk_table(int integ, RKTable &t) {
	std::memset(&t, 0, sizeof t);
	switch (integ) {
	case HYDRO_INT_FORWARD_EULER: t.order = 1; t.a[0][0] = 1; t.b[0][0] = 1; return true;
	case HYDRO_INT_RK2: t.order = 2;
		t.a[0][0] = 1; t.a[1][0] = 1; t.b[0][0] = .5; t.b[1][1] = 1; return true;
	case HYDRO_INT_RK2_HEUN: t.order = 2;
		t.a[0][0] = 1; t.a[1][0] = 1; t.b[0][0] = 1; t.b[1][0] = .5; t.b[1][1] = .5; return true;
	case HYDRO_INT_RK2_RALSTON: t.order = 2;
		t.a[0][0] = 1; t.a[1][0] = 1; t.b[0][0] = 2. / 3.; t.b[1][0] = 1. / 4.; t.b[1][1] = 3. / 4.; return true;
	case HYDRO_INT_RK3: t.order = 3;
		t.a[0][0] = t.a[1][0] = t.a[2][0] = 1;
		t.b[0][0] = .5; t.b[1][0] = -1; t.b[1][1] = 2;
		t.b[2][0] = 1. / 6.; t.b[2][1] = 2. / 6.; t.b[2][2] = 1. / 6.; return true;
	case HYDRO_INT_RK4: t.order = 4;
		for (int i = 0; i < 4; ++i) t.a[i][0] = 1;
		t.b[0][0] = .5; t.b[1][1] = .5; t.b[2][2] = 1;
		t.b[3][0] = 1. / 6.; t.b[3][1] = 2. / 6.; t.b[3][2] = 2. / 6.; t.b[3][3] = 1. / 6.; return true;
	case HYDRO_INT_RK4_3_8THS: t.order = 4;
		for (int i = 0; i < 4; ++i) t.a[i][0] = 1;
		t.b[0][0] = 1. / 3.; t.b[1][0] = -1. / 3.;
		t.b[2][0] = 1; t.b[2][1] = -1; t.b[2][2] = 1;
		t.b[3][0] = 1. / 8.; t.b[3][1] = 3. / 8.; t.b[3][2] = 3. / 8.; t.b[3][3] = 1. / 8.; return true;
	case HYDRO_INT_RK2_TVD: t.order = 2;
		t.a[0][0] = 1; t.a[1][0] = .5; t.a[1][1] = .5; t.b[0][0] = 1; t.b[1][1] = .5; return true;
	case HYDRO_INT_RK2_NON_TVD: t.order = 2;
		t.a[0][0] = 1; t.a[1][0] = 1; t.b[0][0] = -20; t.b[1][0] = 41. / 40.; t.b[1][1] = -1. / 40.; return true;
	case HYDRO_INT_RK3_TVD: t.order = 3;
		t.a[0][0] = 1; t.a[1][0] = 3. / 4.; t.a[1][1] = 1. / 4.; t.a[2][0] = 1. / 3.; t.a[2][2] = 2. / 3.;
		t.b[0][0] = 1; t.b[1][1] = 1. / 4.; t.b[2][2] = 2. / 3.; return true;
	case HYDRO_INT_RK4_TVD: t.order = 4;
		t.a[0][0] = 1;
		t.a[1][0] = 649. / 1600.; t.a[1][1] = 951. / 1600.;
		t.a[2][0] = 53989. / 2500000.; t.a[2][1] = 4806213. / 20000000.; t.a[2][2] = 23619. / 32000.;
		t.a[3][0] = 1. / 5.; t.a[3][1] = 6127. / 30000.; t.a[3][2] = 7873. / 30000.; t.a[3][3] = 1. / 3.;
		t.b[0][0] = .5;
		t.b[1][0] = -10890423. / 25193600.; t.b[1][1] = 5000. / 7873;
		t.b[2][0] = -102261. / 5000000.; t.b[2][1] = -5121. / 20000.; t.b[2][2] = 7873. / 10000.;
		t.b[3][0] = 1. / 10.; t.b[3][1] = 1. / 6.; t.b[3][3] = 1. / 6.; return true;
	case HYDRO_INT_RK4_NON_TVD: t.order = 4;
		for (int i = 0; i < 3; ++i) t.a[i][0] = 1;
		t.a[3][0] = -1. / 3.; t.a[3][1] = 1. / 3.; t.a[3][2] = 2. / 3.; t.a[3][3] = 1. / 3.;
		t.b[0][0] = .5; t.b[1][1] = .5; t.b[2][2] = 1; t.b[3][3] = 1. / 6.; return true;
	}
	return false;
}

static bool needs_deriv(const RKTable &t, int i) {
	for (int m = i + 1; m < t.order; ++m)
		if (t.b[m][i] != 0) return true;
	return false;
}

// ------------------------------------------------------------------ Grid
struct Grid {
	hydro_cfg cfg;
	int dim, Q, NSTAT, S;
	int n[3];
	long ncell;
	long ps;
	size_t elem;
	RKTable rk;
	void *U[4];
	void *D[4];
	void *ping;
	void *stat;
	DevScalars *dev;
	int slot;           // dt slot of the next step
	int dtValid;        // slot holds the min for the current state
	int rowsPerWave;
	int tile;           // plain 2D solver: the tile kernel in place of the marching one
	int wholeSteps;     // plain 1D solver: a launch per step, not per stage
	int nvel;           // Euler: velocity components that are not identically zero
	int wrote;          // the most components any launch has stored since the buffers were clear past nvel
	std::vector<double> ePot;   // Euler ePot of the last upload (dynamics-neutral)
};

static size_t elem_size(const hydro_cfg &c) { return c.precision == HYDRO_REAL_F32 ? 4 : 8; }

static int validate(const hydro_cfg *c) {
	if (!c) return fail("cfg is NULL");
	if (c->dim < 1 || c->dim > 3) return fail("dim %d not supported (1, 2 or 3)", c->dim);
	if (c->dim == 3 && c->eqn != HYDRO_EQN_EULER) return fail("3D is built for the Euler equations only");
	if (c->eqn == HYDRO_EQN_SHALLOW_WATER && !(c->gravity > 0)) return fail("gravity must be > 0");
	for (int i = 0; i < c->dim; ++i)
		if (c->size[i] < 1) return fail("size[%d] = %d must be >= 1", i, c->size[i]);
	if (c->eqn != HYDRO_EQN_EULER && c->eqn != HYDRO_EQN_GLM_MAXWELL && c->eqn != HYDRO_EQN_SHALLOW_WATER)
		return fail("eqn %d not supported", c->eqn);
	if (c->flux < HYDRO_FLUX_ROE || c->flux > HYDRO_FLUX_MARQUINA)
		return fail("flux %d not supported", c->flux);
	if (c->flux != HYDRO_FLUX_ROE && c->eqn != HYDRO_EQN_EULER)
		return fail("the HLL, Rusanov, HLLC and Marquina fluxes take the Euler equations");
	if (c->eqn == HYDRO_EQN_SHALLOW_WATER && c->plm > HYDRO_PLM_CONS)
		return fail("the shallow water equations take 'plm cons' or no reconstruction");
	if (c->roe_entropy_fix && (c->flux != HYDRO_FLUX_ROE || c->eqn != HYDRO_EQN_EULER))
		return fail("the entropy fix belongs to the Roe flux of the Euler equations (roe.cl:83-106)");
	if (c->roe_entropy_fix && !(c->roe_entropy_fix_factor > 0))
		return fail("roe_entropy_fix_factor must be > 0");
	if (c->flux_limiter < 0 || c->flux_limiter >= HYDRO_NUM_LIMITERS) return fail("flux_limiter %d out of range", c->flux_limiter);
	if (c->slope_limiter < 0 || c->slope_limiter >= HYDRO_NUM_LIMITERS) return fail("slope_limiter %d out of range", c->slope_limiter);
	if (c->plm < HYDRO_PLM_NONE || c->plm > HYDRO_PLM_EIG_PRIM_REF)
		return fail("plm %d not supported", c->plm);
	const bool glmPpm = c->plm == HYDRO_PLM_PPM && c->eqn == HYDRO_EQN_GLM_MAXWELL;
	if (c->plm > HYDRO_PLM_CONS && !glmPpm && (c->eqn != HYDRO_EQN_EULER || c->flux != HYDRO_FLUX_ROE || c->roe_entropy_fix))
		return fail("%s is built for the Euler equations with the Roe flux (no entropy fix)",
			c->plm == HYDRO_PLM_PRIM ? "plm prim" : c->plm == HYDRO_PLM_EIG ? "plm eig"
			: c->plm == HYDRO_PLM_CONS_FLUX ? "plm cons with flux" : c->plm == HYDRO_PLM_ATHENA ? "plm athena"
			: c->plm == HYDRO_PLM_PPM ? "ppm" : c->plm == HYDRO_PLM_EIG_PRIM ? "plm eig prim" : "plm eig prim ref");
	// gridsolver.lua:119
	if (c->plm && c->flux_limiter != HYDRO_LIMITER_DONOR_CELL)
		return fail("are you sure you want to use flux and slope limiters at the same time?");
	RKTable t;
	if (!rk_table(c->integrator, t)) return fail("integrator %d not supported", c->integrator);
	for (int f = 0; f < 2 * c->dim; ++f)
		if (c->boundary[f] < 0 || c->boundary[f] > HYDRO_BC_FIXED) return fail("boundary[%d] = %d invalid", f, c->boundary[f]);
	if (c->precision != HYDRO_REAL_F64 && c->precision != HYDRO_REAL_F32) return fail("precision %d invalid", c->precision);
	if (!(c->cfl > 0) && !c->use_fixed_dt) return fail("cfl must be > 0");
	return 0;
}

// Compute units of the current device (256 on MI355X; also when none is found).
static long device_cus() {
	int dev = 0, cus = 0;
	if (hipGetDevice(&dev) != hipSuccess ||
		hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
		return 256;
	return cus;
}

static StageKey stage_key_cfg(const hydro_cfg &cfg, int nvel);

// Blocks of the stage kernel of cfg that a CU holds at once (its registers and
// LDS decide), from an occupancy query: 4 waves a block, or the batched kernel
// with the given waves; 4 if the query fails. The velocity components are taken
// as the dimension's, the usual Euler state.
template <typename R>
static long stage_blocks_per_cu(const hydro_cfg &cfg, int batchWaves) {
	StageArgs<R> a{};
	const StageKey k = stage_key_cfg(cfg, std::min(cfg.dim, 3));
	stage_occupancy = 0;
	if (launch_stage<R>(k, a, dim3(0), dim3(WAVE * batchWaves), nullptr) != hipSuccess || stage_occupancy < 1) {
		(void)hipGetLastError();
		return 4;
	}
	return stage_occupancy;
}
static long stage_occupancy_of(const hydro_cfg &cfg, int batchWaves) {
	return cfg.precision == HYDRO_REAL_F32 ? stage_blocks_per_cu<float>(cfg, batchWaves)
	                                       : stage_blocks_per_cu<double>(cfg, batchWaves);
}

// The marching kernel's time, but for a constant: L waves for each SIMD, of which
// it holds occ at once, march `rows` (warm-up and edge pass included) each. k
// waves together take 3 + k where one takes 4: a row is a chain of dependent
// loads, square roots and divisions, and one wave alone fills a quarter of its
// SIMD. (Measured, a row of FP32 'plm cons': 2.0, 2.65, 3.1, 3.4 us for 1..4
// waves.) alone is that 3; 2 for the IEEE kernels of which a SIMD holds two waves at
// most, whose division sequences fill more of it (march_alone).
static double march_cost(long L, long occ, double rows, double alone = 3.) {
	const long rem = L % occ;
	return rows * ((double)(L / occ) * (alone + (double)occ) + (rem ? alone + (double)rem : 0.));
}
// IEEE FP64 640x480, us per stage at 3 rows (two waves a SIMD) and 5 (one): 'plm athena' 46.0
// and 40.9, 'plm eig prim' 45.5 and 40.2, 'plm eig prim ref' 48.9 and 41.6. Over 29 such cases
// of 420x380 .. 1500x1100 the rows taken are within 1.9 % of the best (17 % at 3), over
// the 117 others, of more waves a SIMD, at 3 within 6.5 % (18 % at 2).
static double march_alone(const hydro_cfg &cfg, long occ) { return !cfg.fast_math && occ <= 2 ? 2. : 3.; }

// Rows a wave marches before or beside its own: the warm-up, and in the
// 64-column strips the edge pass, about 1.5 rows of work (.5 where four waves of
// a block share one); the first loads of the equations with a source, of more
// fields, are about 1.2 rows' time (GLM-Maxwell FP32 512^2: 13.6 us at 3 rows, 14.3
// at 2).
static double march_overhead(const hydro_cfg &cfg, bool shared) {
	const int warm = cfg.plm ? 2 : (cfg.flux_limiter ? 3 : 1);
	const bool edges = strip_edges(cfg.dim, eqn_has_source(cfg.eqn));
	return warm + (!edges ? 1.2 : shared ? .5 : 1.5);
}

static long grid_strips(const hydro_cfg &cfg) {
	const int so = strip_out(strip_edges(cfg.dim, eqn_has_source(cfg.eqn)));
	return (cfg.size[0] + so - 1) / so;
}

// Rows per wave of the plain marching kernel: in 2D those in 2..8 of the least
// march_cost. Short waves fill a grid that leaves SIMDs idle, long ones save
// warm-ups, and the last round of waves should be a full one; beyond 8 nothing
// is gained at 2048^2 and 4096^2, but a kernel of at most 3 blocks per CU
// takes up to 16, so that its launch can end in fewer rounds (GLM-Maxwell FP64: 10
// rows at 1024^2, 12 at 2048^2; at 1500x1100 IEEE 'plm cons' 9 rows 93 us, 7 103,
// HLLC 56 and 60, 'plm eig prim' 89 and 95, shallow water 10 rows 54.4, 5 57). us per stage at the rows
// taken (against 4..8 by an older fit): shallow water 700x500 17.5 (19.3),
// GLM-Maxwell FP32 512^2 14.3 (15.1), 700^2 17.4 (19.6), KH FP64 700^2 19.3 (23.5);
// over 26 uneven shapes of all equations the rows taken were within 4 % of the
// best of 2..16, most of them the best.
// 3D: planes per block chunk, by the same cost over blocks of four waves; the
// warm-up (reconstruction or jumps and one flux) and the edge pass are a plane's
// work together. FP32 takes 2..8, FP64, with fewer blocks resident and a larger
// state, 2..16: at 256^3 FP32 stages take 505 us at 8 planes and 515 at 16, FP64
// 1027 and 993. us at the planes taken (against 8 at least, by an older rule):
// 64^3 FP32 19.1 (32.7), FP64 24.8 (36.8); 128^3 FP32 76 (78); 180^3 FP64 381 (406).
static int default_rows(const hydro_cfg &cfg) {
	if (cfg.dim < 2) return 1;
	const long stripsX = grid_strips(cfg), ny = cfg.size[1];
	const long cus = device_cus(), occ = stage_occupancy_of(cfg, 0);
	int best = 2;
	double bestT = -1;
	if (cfg.dim == 3) {
		const bool f32 = cfg.precision == HYDRO_REAL_F32;
		const long W = f32 ? Block3<float>::W : Block3<double>::W;
		const long perPlane = stripsX * ((ny + W - 1) / W);
		for (int r = 2; r <= (f32 ? EDGE_PLANES / 2 : EDGE_PLANES); ++r) {
			const long blocks = perPlane * ((cfg.size[2] + r - 1) / r);
			const double t = march_cost((blocks + cus - 1) / cus, occ, r + 1.);
			if (bestT < 0 || t < bestT * (1 - 1e-9)) { best = r; bestT = t; }
		}
		return best;
	}
	const int rMax = occ <= 3 ? 16 : 8;
	for (int r = 2; r <= rMax; ++r) {
		const long blocks = (stripsX * ((ny + r - 1) / r) + 3) / 4;
		const double t = march_cost((blocks + cus - 1) / cus, occ,
			r + march_overhead(cfg, stripsX % 4 == 0 && 5 * r <= WAVE), march_alone(cfg, occ));
		if (bestT < 0 || t < bestT * (1 - 1e-9)) { best = r; bestT = t; }
	}
	return best;
}

// Rows per wave of a batched launch over 2D grids of one configuration: by the
// same cost, 2..32 rows. waves: of a block, perCU: such blocks resident on a CU.
// Within 5 % of the best of 2..32 on ensembles of 4 to 64 grids, both precisions;
// us per stage (at rows from the mean load): 48 FP32 grids of 64..512 78 (95), 24
// 47 (61), 24 GLM-Maxwell FP32 33 (45), 24 FP64 62 (90).
static int batch_rows(const std::vector<const hydro_cfg *> &grids, int waves, long perCU) {
	const hydro_cfg &cfg = *grids[0];
	if (cfg.dim < 2) return 1;
	const long simds = 4 * (long)device_cus(), occ = std::max(1L, perCU * waves / 4);
	int best = 2;
	double bestT = -1;
	for (int r = 2; r <= EDGE_ROWS; ++r) {
		long items = 0;
		for (const hydro_cfg *c : grids) items += grid_strips(*c) * ((c->size[1] + r - 1) / r);
		const double t = march_cost((items + simds - 1) / simds, occ, r + march_overhead(cfg, false));
		if (bestT < 0 || t < bestT * (1 - 1e-9)) { best = r; bestT = t; }
	}
	return best;
}

// The tile kernel's strips (its blocks per TILE_W rows) and blocks on a 2D grid.
static int tile_strips(const hydro_cfg &cfg) {
	const bool lim = cfg.plm == HYDRO_PLM_NONE && cfg.flux == HYDRO_FLUX_ROE && cfg.flux_limiter != HYDRO_LIMITER_DONOR_CELL;
	const int so = strip_out(tile_edges(eqn_has_source(cfg.eqn), lim));
	return (cfg.size[0] + so - 1) / so;
}
static long tile_blocks(const hydro_cfg &cfg) {
	return (long)tile_strips(cfg) * ((cfg.size[1] + TILE_W - 1) / TILE_W);
}

// Whether the plain 2D solver takes the tile kernel (fv_tile.h) and not the
// marching one. Its time is about 5.2 us plus 1.4-1.8 us (IEEE 3) for each block
// a CU has to run; the marching kernel's is flat (FAST 9-14 us at 2 or 3 rows, IEEE
// 22-35 us, by the scheme) while its waves are all resident at once and then grows at
// half to two thirds of that rate. Measured at 4 blocks per CU (384^2), tile /
// marching at its best rows: 'plm cons' FP64 10.6 / 12.5, FP32 9.3 / 10.6, van Leer
// 10.1 / 12.0, flux-limited 11.7 / 14.0, shallow water 11.5 / 12.1, GLM-Maxwell FP32
// 10.6 / 10.7; at 256^2 7.8 / 10.6, 7.2 / 9.7, 7.8 / 10.7, 8.6 / 12.0, 8.1 / 9.5,
// 7.4 / 8.8; 'plm cons' at 5.3 (512^2) 15.0 / 14.8. GLM-Maxwell FP64, twelve state
// components in 64 bits, 8.9 / 9.9 at 1.7 (256^2), 10.8 / 10.5 at 2.5 (320^2). IEEE at
// 14 (about 830^2): 47.1 / 50.9 at 800^2, but 'plm athena' 44.6 / 40.6 at 640x480.
static bool tile_form(const hydro_cfg &cfg) {
	if (cfg.dim != 2) return false;
	const bool heavy = cfg.eqn == HYDRO_EQN_GLM_MAXWELL && cfg.precision == HYDRO_REAL_F64;
	const bool cons = cfg.plm == HYDRO_PLM_NONE || cfg.plm == HYDRO_PLM_CONS;
	const double perCU = !cfg.fast_math && cons ? 14. : heavy ? 2.4 : 4.5;
	return (double)tile_blocks(cfg) <= perCU * (double)device_cus();
}

static void grid_init(Grid &g, const hydro_cfg &cfg) {
	g.cfg = cfg;
	g.dim = cfg.dim;
	g.Q = num_int_states(cfg.eqn);
	g.S = num_states(cfg.eqn);
	g.NSTAT = num_static_states(cfg.eqn);
	g.ncell = 1;
	for (int i = 0; i < 3; ++i) {
		g.n[i] = i < g.dim ? cfg.size[i] : 1;
		g.ncell *= g.n[i];
	}
	g.ps = g.ncell;
	g.elem = elem_size(cfg);
	rk_table(cfg.integrator, g.rk);
	std::memset(g.U, 0, sizeof g.U);
	std::memset(g.D, 0, sizeof g.D);
	g.ping = g.stat = nullptr;
	g.dev = nullptr;
	g.slot = 0;
	g.dtValid = 0;
	g.nvel = 3;
	g.wrote = 0;
	g.rowsPerWave = 1;       // the caller's to set, as the form is
	g.tile = 0;
	g.wholeSteps = 0;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// device bytes of a grid, in the order grid_bind lays them out
static size_t grid_bytes(const Grid &g) {
	size_t plane = (size_t)g.ps * g.elem, state = align256(plane * g.Q);
	size_t b = align256(sizeof(DevScalars));
	int o = g.rk.order;
	for (int i = 0; i < o; ++i) {
		b += state;
		if (needs_deriv(g.rk, i)) b += state;
	}
	if (o == 1) b += state;
	if (g.NSTAT) b += align256(plane * g.NSTAT);
	return b;
}

static void grid_bind(Grid &g, char *base) {
	size_t plane = (size_t)g.ps * g.elem, state = align256(plane * g.Q);
	char *p = base;
	g.dev = (DevScalars *)p;
	p += align256(sizeof(DevScalars));
	int o = g.rk.order;
	for (int i = 0; i < o; ++i) {
		g.U[i] = p;
		p += state;
		if (needs_deriv(g.rk, i)) {
			g.D[i] = p;
			p += state;
		}
	}
	if (o == 1) {
		g.ping = p;
		p += state;
	}
	if (g.NSTAT) {
		g.stat = p;
		p += align256(plane * g.NSTAT);
	}
}

// zero every state buffer, +inf every dt slot (asynchronous on s)
[[maybe_unused]] static int grid_clear(Grid &g, char *base, hipStream_t s) {
	HIPCHECK(hipMemsetAsync(base, 0, grid_bytes(g), s));
	DevScalars z;
	std::memset(&z, 0, sizeof z);
	for (int i = 0; i < 3; ++i)
		for (int j = 0; j < DT_LANES; ++j) z.dtmin[i][j] = INFINITY;
	HIPCHECK(hipMemcpyAsync(g.dev, &z, sizeof z, hipMemcpyHostToDevice, s));
	return 0;
}

// The stage kernels store no momentum past g.nvel, and an upload writes U[0] alone:
// where steps end in another buffer that then becomes U[0] (forward Euler, whole 1D
// steps), that buffer's planes past nvel still hold what a state with more
// components left there. Clears them, once per upload that has fewer.
[[maybe_unused]] static int clear_past_nvel(Grid &g, hipStream_t s) {
	if (g.wrote <= g.nvel) return 0;
	const size_t plane = (size_t)g.ps * g.elem;
	void *other = g.ping ? g.ping : g.wholeSteps ? g.U[1] : nullptr;
	if (other)
		HIPCHECK(hipMemsetAsync((char *)other + (1 + g.nvel) * plane, 0, (g.wrote - g.nvel) * plane, s));
	g.wrote = g.nvel;
	return 0;
}

static CflScale cfl_scale(const Grid &g) {
	CflScale s;
	s.len = INFINITY;
	for (int i = 2; i >= 0; --i) {
		s.dx[i] = (g.cfg.maxs[i] - g.cfg.mins[i]) / (double)g.n[i];
		if (i < g.dim && s.dx[i] > 0.) s.len = s.dx[i];
	}
	for (int i = 0; i < 3; ++i) s.scale[i] = i < g.dim && s.dx[i] > 0. ? s.len / s.dx[i] : 0.;
	return s;
}

template <typename R>
static void grid_desc(const Grid &g, GridDesc<R> &d) {
	std::memset(&d, 0, sizeof d);
	for (int i = 0; i < 4; ++i) {
		d.U[i] = (R *)g.U[i];
		d.D[i] = (R *)g.D[i];
	}
	d.ping = (R *)g.ping;
	d.stat = (const R *)g.stat;
	for (int i = 0; i < 3; ++i) d.n[i] = g.n[i];
	d.ps = g.ps;
	d.step1 = g.n[0];
	const hydro_cfg &c = g.cfg;
	for (int f = 0; f < 6; ++f) {
		d.bc[f] = c.boundary[f];
		for (int j = 0; j < g.Q + g.NSTAT; ++j) d.fixedv[f][j] = R(c.boundary_fixed[f][j]);
	}
	// fvsolver.cl:37-102 in the stored precision: volume = 1 * dx0 * dx1...,
	// areaL = 1 * prod(dx_other), areaL *= 1 / volume
	R dxr[3];
	for (int i = 0; i < 3; ++i) {
		dxr[i] = R((c.maxs[i] - c.mins[i]) / (double)g.n[i]);
		d.dx[i] = dxr[i];
		d.invdx[i] = R(1) / dxr[i];
		d.inv2dx[i] = R(1) / (dxr[i] * R(2));
	}
	d.cflScale = cfl_scale(g);
	R volume = R(1);
	for (int i = 0; i < g.dim; ++i) volume = volume * dxr[i];
	d.derivOn = volume > R(1e-7);
	R invVolume = R(1) / volume;
	for (int side = 0; side < 3; ++side) {
		R area = R(1);
		for (int i = 0; i < g.dim; ++i)
			if (i != side) area = area * dxr[i];
		R aL = area;
		if (aL <= R(1e-7)) aL = R(0);
		d.areaOverVol[side] = aL * invVolume;
		d.fluxOn[side] = area > R(1e-7);
		// both guards as one factor: the flux term is then exactly 0 where a
		// guard is off (for finite fluxes; the sign of a zero may differ)
		d.aovFast[side] = d.fluxOn[side] && d.derivOn ? d.areaOverVol[side] : R(0);
		d.aovHalf[side] = R(.5) * d.aovFast[side];
	}
	d.cfl = c.cfl;
	d.rowsPerWave = g.rowsPerWave;
	const int so = strip_out(strip_edges(g.dim, eqn_has_source(g.cfg.eqn)));
	d.stripsX = (g.n[0] + so - 1) / so;
	if (g.dim == 3) {
		d.stripsY = (g.n[1] + Block3<R>::W - 1) / Block3<R>::W;
		d.stripsZ = (g.n[2] + g.rowsPerWave - 1) / g.rowsPerWave;
	} else {
		d.stripsY = g.dim >= 2 ? (g.n[1] + g.rowsPerWave - 1) / g.rowsPerWave : 1;
		d.stripsZ = 1;
	}
	d.nItems = (long)d.stripsX * d.stripsY * d.stripsZ;
	d.active = 1;
	d.itemBase = 0;
	d.dev = g.dev;
	d.stepsLeft = 1 << 30;
}

// Uniform arguments of stage s (0-based) of the table.
template <typename R>
static void stage_args(const Grid &g, int s, StageArgs<R> &a) {
	std::memset(&a, 0, sizeof a);
	const RKTable &t = g.rk;
	int o = t.order;
	a.src = s;
	bool last = s == o - 1;
	a.out = !last ? s + 1 : (o == 1 ? -1 : 0);
	a.nAlpha = 0;
	for (int k = 0; k <= s; ++k) {
		if (t.a[s][k] != 0) {
			a.accU[a.nAlpha] = k;
			a.alpha[a.nAlpha] = t.a[s][k];
			a.nAlpha++;
		}
	}
	a.nStoredD = 0;
	for (int k = 0; k < s; ++k) {
		if (t.b[s][k] != 0) {
			a.accD[a.nStoredD] = k;
			a.beta[a.nStoredD] = t.b[s][k];
			a.nStoredD++;
		}
	}
	a.storeD = needs_deriv(t, s) ? s : -1;
	a.betaNew = t.b[s][s];
	a.steps = 0;
	const hydro_cfg &c = g.cfg;
	a.gamma = R(c.gamma);
	a.rhoMin = R(c.rho_min);
	a.PMin = R(c.P_min);
	a.divPhi = R(c.div_phi_wavespeed);
	a.divPsi = R(c.div_psi_wavespeed);
	a.gravity = R(c.gravity);
	a.pd = eqn_par_d(c);
	a.roeFixFactor = R(c.roe_entropy_fix_factor);
	a.limiter = c.plm ? c.slope_limiter : c.flux_limiter;
	a.resetSlot = -1;
	a.reduceSlot = -1;
	a.dtSlot = -1;
	a.advanceTime = 0;
	a.xcdRemap = 1;
	a.shareEdges = 0;
	a.tile = 0;
}

static StageKey stage_key_cfg(const hydro_cfg &cfg, int nvel) {
	StageKey k;
	k.eqn = cfg.eqn;
	k.dim = cfg.dim;
	k.plm = cfg.plm != HYDRO_PLM_NONE;
	k.flux = cfg.flux;
	k.roeFix = cfg.roe_entropy_fix != 0;
	k.plmKind = cfg.plm;
	// only the Roe flux uses a flux limiter (fvsolver.lua:63)
	k.lim = !k.plm && k.flux == HYDRO_FLUX_ROE && cfg.flux_limiter != HYDRO_LIMITER_DONOR_CELL;
	k.limiter = k.plm ? cfg.slope_limiter : cfg.flux_limiter;
	k.fast = cfg.fast_math != 0;
	k.nvel = nvel;
	return k;
}

static StageKey stage_key(const Grid &g) { return stage_key_cfg(g.cfg, g.nvel); }

// ------------------------------------------------------- layout conversion
// Ghost coordinate -> interior source, following the reference's x, y, z
// boundary passes (gridsolver.lua:1272-1314).
struct HostMap {
	int idx, mirror, fixedFace;
};
static HostMap host_map(int c, int n, int kmin, int kmax, int faceMin) {
	HostMap m{c, 0, -1};
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
	m.idx = std::max(0, std::min(n - 1, m.idx));
	return m;
}

static bool reflects(int eqn, int field, int axis) {
	if (eqn == HYDRO_EQN_EULER || eqn == HYDRO_EQN_SHALLOW_WATER) return field == 1 + axis;
	return field == axis || field == 3 + axis;
}

static size_t ghosted_cells(const Grid &g) {
	size_t c = 1;
	for (int i = 0; i < 3; ++i) c *= (size_t)(i < g.dim ? g.n[i] + 2 * NG : 1);
	return c;
}

// Runs fn(r0, r1) over [0, n) split into contiguous ranges on up to 8 host
// threads (one range, on the caller's thread, below `grain` items).
template <typename F>
static void parallel_ranges(long n, long grain, F fn) {
	const long hw = std::max(1L, (long)std::thread::hardware_concurrency());
	const long nt = std::max(1L, std::min({8L, hw, n / std::max(1L, grain)}));
	if (nt <= 1) {
		fn(0L, n);
		return;
	}
	std::vector<std::thread> th;
	th.reserve(nt - 1);
	for (long t = 1; t < nt; ++t) th.emplace_back(fn, n * t / nt, n * (t + 1) / nt);
	fn(0L, n / nt);
	for (auto &x : th) x.join();
}

// AoS ghosted cons_t -> the device layout (q planes and nstat static planes of
// ps values each, interior cells dense, the rest zero), into host memory the
// caller provides; sets g.nvel and g.ePot from the state. Rows are packed on
// several host threads.
template <typename R>
static void pack_interior(Grid &g, const R *aos, R *planes, R *stat) {
	int gs[3], o[3];
	for (int i = 0; i < 3; ++i) {
		gs[i] = i < g.dim ? g.n[i] + 2 * NG : 1;
		o[i] = i < g.dim ? NG : 0;
	}
	const bool euler = g.cfg.eqn == HYDRO_EQN_EULER;
	if (euler) g.ePot.assign(g.ncell, 0.);
	const long rows = (long)g.n[1] * g.n[2];
	const int nx = g.n[0], Q = g.Q, NS = g.NSTAT, S = g.S, dim = g.dim;
	const long ps = g.ps;
	double *ePot = euler ? g.ePot.data() : nullptr;
	// per-row flags (each row written by one thread), reduced afterwards
	std::vector<char> rowE(euler ? rows : 0, 0), rowV(euler ? rows : 0, 0);
	parallel_ranges(rows, 64, [&](long r0, long r1) {
		for (long row = r0; row < r1; ++row) {
			const int j = (int)(row % g.n[1]), k = (int)(row / g.n[1]);
			const R *u = aos + ((size_t)o[0] + (size_t)gs[0] * ((j + o[1]) + (size_t)gs[1] * (k + o[2]))) * S;
			const size_t c0 = (size_t)nx * (size_t)row;
			bool anyE = false, nzv = false;
			for (int i = 0; i < nx; ++i, u += S) {
				const size_t c = c0 + i;
				for (int f = 0; f < Q; ++f) planes[(size_t)f * ps + c] = u[f];
				for (int f = 0; f < NS; ++f) stat[(size_t)f * ps + c] = u[Q + f];
				if (euler) {
					ePot[c] = (double)u[5];
					anyE = anyE || u[5] != R(0);
					for (int f = 1 + dim; f <= 3; ++f) nzv = nzv || u[f] != R(0);
				}
			}
			if (euler) {
				rowE[row] = anyE;
				rowV[row] = nzv;
			}
		}
	});
	// each plane's cells past the interior (none while the planes are dense)
	for (int f = 0; f < Q; ++f) std::fill(planes + (size_t)f * ps + g.ncell, planes + (size_t)(f + 1) * ps, R(0));
	for (int f = 0; f < NS; ++f) std::fill(stat + (size_t)f * ps + g.ncell, stat + (size_t)(f + 1) * ps, R(0));
	bool anyE = false, nzv = false;
	for (long r = 0; r < (long)rowE.size(); ++r) {
		anyE = anyE || rowE[r];
		nzv = nzv || rowV[r];
	}
	if (!anyE) g.ePot.clear();
	// Euler: momentum components beyond dim that are zero everywhere stay zero
	// (their fluxes and wave amplitudes are exact zeros), so the kernels skip them
	g.nvel = euler && dim < 3 && !nzv ? dim : 3;
}

template <typename R>
static void unpack_with_ghosts(const Grid &g, const R *planes, const R *stat, R *aos) {
	int gs[3];
	for (int i = 0; i < 3; ++i) gs[i] = i < g.dim ? g.n[i] + 2 * NG : 1;
	const hydro_cfg &c = g.cfg;
	parallel_ranges((long)gs[1] * gs[2], 64, [&](long r0, long r1) {
		for (long row = r0; row < r1; ++row) {
			const int j = (int)(row % gs[1]), k = (int)(row / gs[1]);
			for (int i = 0; i < gs[0]; ++i) {
				int cc[3] = {i - (g.dim > 0 ? NG : 0), j - (g.dim > 1 ? NG : 0), k - (g.dim > 2 ? NG : 0)};
				HostMap m[3];
				for (int a = 0; a < 3; ++a) {
					if (a < g.dim) m[a] = host_map(cc[a], g.n[a], c.boundary[2 * a], c.boundary[2 * a + 1], 2 * a);
					else m[a] = HostMap{0, 0, -1};
				}
				size_t src = (size_t)m[0].idx + (size_t)g.n[0] * (m[1].idx + (size_t)g.n[1] * m[2].idx);
				R *u = aos + ((size_t)i + (size_t)gs[0] * (j + (size_t)gs[1] * k)) * g.S;
				for (int f = 0; f < g.S; ++f) {
					R v;
					if (f < g.Q) v = planes[(size_t)f * g.ps + src];
					else if (f - g.Q < g.NSTAT) v = stat[(size_t)(f - g.Q) * g.ps + src];
					else v = (g.cfg.eqn == HYDRO_EQN_EULER && !g.ePot.empty()) ? R(g.ePot[src]) : R(0);
					for (int a = 0; a < g.dim; ++a) {
						if (m[a].fixedFace >= 0) v = R(c.boundary_fixed[m[a].fixedFace][f]);
						else if (m[a].mirror && reflects(c.eqn, f, a)) v = -v;
					}
					u[f] = v;
				}
			}
		}
	});
}

template <typename R>
static GridArgs<R> grid_args(const Grid &g, int slot) {
	GridArgs<R> a;
	std::memset(&a, 0, sizeof a);
	a.U = (R *)g.U[0];
	a.stat = (const R *)g.stat;
	a.ps = g.ps;
	a.ncell = g.ncell;
	a.dim = g.dim;
	a.cflScale = cfl_scale(g);
	a.pd = eqn_par_d(g.cfg);
	a.dev = g.dev;
	a.slot = slot;
	return a;
}

static int grid_dt_kernel(Grid &g, int slot, hipStream_t s) {
	HIPCHECK(launch_reset_slots(g.dev, 1 << slot, s));
	hipError_t e = g.elem == 8 ? launch_dt<double>(g.cfg.eqn, g.dim, g.cfg.fast_math, grid_args<double>(g, slot), s)
	                           : launch_dt<float>(g.cfg.eqn, g.dim, g.cfg.fast_math, grid_args<float>(g, slot), s);
	if (e != hipSuccess) return fail("dt kernel: %s", hipGetErrorString(e));
	return 0;
}

[[maybe_unused]] static int grid_constrain(Grid &g, hipStream_t s) {
	hipError_t e = g.elem == 8 ? launch_constrain<double>(g.cfg.eqn, g.cfg.fast_math, grid_args<double>(g, 0), s)
	                           : launch_constrain<float>(g.cfg.eqn, g.cfg.fast_math, grid_args<float>(g, 0), s);
	if (e != hipSuccess) return fail("constrainU kernel: %s", hipGetErrorString(e));
	g.dtValid = 0;
	return 0;
}

[[maybe_unused]] static int grid_calc_dt(Grid &g, double *dt, hipStream_t s) {
	if (g.cfg.use_fixed_dt) { *dt = g.cfg.fixed_dt; return 0; }
	if (grid_dt_kernel(g, g.slot, s)) return -1;
	HIPCHECK(launch_fold_slot(g.dev, g.slot, s));
	double m;
	HIPCHECK(hipMemcpyAsync(&m, &g.dev->dtmin[g.slot][0], sizeof m, hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	g.dtValid = 1;
	*dt = g.cfg.cfl * m;
	return 0;
}

[[maybe_unused]] static int grid_get_time(const Grid &g, double *t, double *dt, hipStream_t s) {
	double v[2];
	HIPCHECK(hipMemcpyAsync(v, &g.dev->t, sizeof v, hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	if (t) *t = v[0];
	if (dt) *dt = v[1];
	return 0;
}

[[maybe_unused]] static int grid_set_time(Grid &g, double t, hipStream_t s) {
	HIPCHECK(hipMemcpyAsync(&g.dev->t, &t, sizeof t, hipMemcpyHostToDevice, s));
	HIPCHECK(hipStreamSynchronize(s));
	return 0;
}


// One stage of every grid described by descs (device array of nGrids
// GridDesc), as one persistent launch. rep supplies the shared configuration.
template <typename R>
static int launch_batched_stage(const Grid &rep, int nvel, int s, int cur, const GridDesc<R> *descs, int nGrids,
	long totalItems, int stepInTick, int wavesPerBlock, int xcdRemap, hipStream_t stream)
{
	int o = rep.rk.order;
	int fixed = rep.cfg.use_fixed_dt;
	bool last = s == o - 1;
	StageArgs<R> a;
	stage_args<R>(rep, s, a);
	if (!fixed) a.dtSlot = cur;
	else a.hostDt = rep.cfg.fixed_dt;
	a.resetSlot = (!fixed && s == 0) ? (cur + 2) % 3 : -1;
	a.reduceSlot = (!fixed && last) ? (cur + 1) % 3 : -1;
	a.advanceTime = last;
	a.stepInTick = stepInTick;
	a.grids = descs;
	a.nGrids = nGrids;
	a.totalItems = totalItems;
	a.xcdRemap = xcdRemap;
	StageKey k = stage_key(rep);
	k.nvel = nvel;
	hipError_t e = launch_stage<R>(k, a, dim3(0), dim3(64 * wavesPerBlock), stream);
	if (e != hipSuccess) return fail("batched stage launch: %s", hipGetErrorString(e));
	return 0;
}

} // namespace hydro
