// fv_aux.h — the small kernels around the fused stage: standalone calcDT with
// its min-reduction, constrainU, dt-slot reset, and deterministic compensated
// conserved-total sums.
#pragma once

#include "fv_common.h"
#include "fv_euler.h"
#include "fv_glm.h"

namespace hydro {

// Shape of the interior state for the elementwise kernels.
template <typename R>
struct GridArgs {
	R *U;            // q integrated planes
	const R *stat;   // static planes
	long ps;         // plane stride
	long ncell;      // interior cells (planes are dense)
	int dim;
	CflScale cflScale;
	EqnParD pd;
	DevScalars *dev;
	int slot;
};

[[maybe_unused]] static __global__ void reset_slots_kernel(DevScalars *dev, int mask) {
	if (blockIdx.x == 0 && threadIdx.x < DT_LANES) {
		for (int i = 0; i < 3; ++i)
			if (mask & (1 << i)) dev->dtmin[i][threadIdx.x] = INFINITY;
	}
}

// min of the 64 sub-slots into sub-slot 0 (for host readback)
[[maybe_unused]] static __global__ void fold_slot_kernel(DevScalars *dev, int slot) {
	double m = read_dt_slot(dev, slot);
	if (threadIdx.x == 0) dev->dtmin[slot][0] = m;
}

// Whether any stored value of a state is not finite: the q integrated and the
// nstat static planes over the interior cells. Sets *flag to 1 and never
// clears it (the caller starts it at 0).
template <typename R>
__global__ void __launch_bounds__(256) nonfinite_kernel(const R *U, const R *stat, long ps, long ncell, int q,
	int nstat, unsigned *flag)
{
	bool bad = false;
	for (int f = 0; f < q + nstat; ++f) {
		const R *p = f < q ? U + (long)f * ps : stat + (long)(f - q) * ps;
		for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += (long)gridDim.x * blockDim.x)
			bad = bad || !__builtin_isfinite(p[c]);
	}
	if (wave_any(bad) && (threadIdx.x & 63) == 0) atomicOr(flag, 1u);
}

// ------------------------------------------------------------ host transfers
// The reference's ghosted cons_t buffer (cells of S reals, x fastest) against the
// planes of the interior, one pinned chunk of consecutive cells at a time. The
// chunk lives in host memory that the kernel addresses directly, so the bus is
// crossed once, in 16-byte pieces of consecutive lanes; the transpose between
// cells and planes goes through LDS. Bound by the bus (about 50 GB/s; 3.2 MB of a
// 256^2 FP64 state in 70 us).
template <typename R>
struct CellBuffer {
	R *U;                 // q integrated planes
	R *stat;              // static planes
	long ps;
	int n[3], dim;
	int q, nstat, S;      // planes, and reals per cell of the buffer
	int bc[6];
	R fixedv[6][HYDRO_MAX_STATES];
	int vec1, vec2;       // first fields of the vectors a mirror reflects (euler: 1; GLM: 0 and 3), -1 none
	R *cells;             // the chunk, in pinned host memory
	long first, count;    // its cells, numbered over the ghosted buffer
	int *flags;           // take_cells: [0] a real past the planes is not 0, [1] an out-of-plane momentum is not 0
};
constexpr int CELLS_BLOCK = 256;

// ghosted coordinates of cell c
template <typename R>
__device__ __forceinline__ void cell_coords(const CellBuffer<R> &b, long c, int *cc) {
	const int gx = b.n[0] + 2 * NG;
	const int gy = b.dim > 1 ? b.n[1] + 2 * NG : 1;
	const long row = c / gx;
	cc[0] = (int)(c - row * gx) - NG;
	cc[2] = (int)(row / gy) - (b.dim > 2 ? NG : 0);
	cc[1] = (int)(row % gy) - (b.dim > 1 ? NG : 0);
}

// planes -> cells, ghosts filled as after the reference's boundary() (axis by
// axis, a later axis wins)
template <typename R>
__global__ void __launch_bounds__(CELLS_BLOCK) give_cells_kernel(const CellBuffer<R> b) {
	__shared__ __align__(16) R sh[CELLS_BLOCK * HYDRO_MAX_STATES];
	const long base = (long)blockIdx.x * CELLS_BLOCK;
	const int here = (int)min((long)CELLS_BLOCK, b.count - base);
	const int t = threadIdx.x;
	if (t < here) {
		int cc[3];
		cell_coords(b, b.first + base + t, cc);
		Mapped m[3];
#pragma unroll
		for (int a = 0; a < 3; ++a) {
			if (a < b.dim) m[a] = map_coord(cc[a], b.n[a], b.bc[2 * a], b.bc[2 * a + 1], 2 * a);
			else { m[a].idx = 0; m[a].mirror = 0; m[a].fixedFace = -1; }
		}
		const long src = (long)m[0].idx + (long)b.n[0] * (m[1].idx + (long)b.n[1] * m[2].idx);
		for (int f = 0; f < b.S; ++f) {
			R v = f < b.q ? b.U[f * b.ps + src] : f < b.q + b.nstat ? b.stat[(f - b.q) * b.ps + src] : R(0);
#pragma unroll
			for (int a = 0; a < 3; ++a) {
				if (m[a].fixedFace >= 0) v = b.fixedv[m[a].fixedFace][f];
				else if (m[a].mirror && (f == b.vec1 + a || (b.vec2 >= 0 && f == b.vec2 + a))) v = -v;
			}
			sh[t * b.S + f] = v;
		}
	}
	__syncthreads();
	const int reals = here * b.S;
	constexpr int PER = 16 / sizeof(R);
	R *out = b.cells + base * b.S;     // 16-byte aligned: CELLS_BLOCK cells are a multiple of 16 bytes
	for (int i = t * PER; i < reals; i += CELLS_BLOCK * PER) {
		if (i + PER <= reals) {
			*(int4 *)(out + i) = *(const int4 *)(sh + i);
		} else {
			for (int k = i; k < reals; ++k) out[k] = sh[k];
		}
	}
}

// cells -> planes, interior cells only
template <typename R>
__global__ void __launch_bounds__(CELLS_BLOCK) take_cells_kernel(const CellBuffer<R> b) {
	__shared__ __align__(16) R sh[CELLS_BLOCK * HYDRO_MAX_STATES];
	const long base = (long)blockIdx.x * CELLS_BLOCK;
	const int here = (int)min((long)CELLS_BLOCK, b.count - base);
	const int t = threadIdx.x;
	const int reals = here * b.S;
	constexpr int PER = 16 / sizeof(R);
	const R *in = b.cells + base * b.S;
	for (int i = t * PER; i < reals; i += CELLS_BLOCK * PER) {
		if (i + PER <= reals) {
			*(int4 *)(sh + i) = *(const int4 *)(in + i);
		} else {
			for (int k = i; k < reals; ++k) sh[k] = in[k];
		}
	}
	__syncthreads();
	bool past = false, outOfPlane = false;
	if (t < here) {
		int cc[3];
		cell_coords(b, b.first + base + t, cc);
		bool inside = true;
#pragma unroll
		for (int a = 0; a < 3; ++a)
			if (a < b.dim) inside = inside && cc[a] >= 0 && cc[a] < b.n[a];
		if (inside) {
			const long dst = (long)cc[0] + (long)b.n[0] * (cc[1] + (long)b.n[1] * cc[2]);
			for (int f = 0; f < b.S; ++f) {
				const R v = sh[t * b.S + f];
				if (f < b.q) b.U[f * b.ps + dst] = v;
				else if (f < b.q + b.nstat) b.stat[(f - b.q) * b.ps + dst] = v;
				else past = past || v != R(0);
				if (f >= 1 + b.dim && f <= 3) outOfPlane = outOfPlane || v != R(0);
			}
		}
	}
	// every wave that found one writes the same 1
	if (wave_any(past) && (t & 63) == 0) b.flags[0] = 1;
	if (wave_any(outOfPlane) && (t & 63) == 0) b.flags[1] = 1;
}

// calcDT (eqn.lua:1187-1224 + calcDT.cl:38-73) and reduceMin: per-cell dt in
// double, wave min, one atomic min per wave into dev->dtmin[slot].
template <typename R, template <typename> class EQ, int DIM>
__global__ void __launch_bounds__(256) dt_kernel(const GridArgs<R> g) {
	using E = EQ<R>;
	constexpr int Q = E::Q;
	FastestOf<R, E, DIM> fw;
	for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long)gridDim.x * blockDim.x) {
		double u[Q + E::NSTAT];
#pragma unroll
		for (int j = 0; j < Q; ++j) u[j] = (double)g.U[j * g.ps + c];
#pragma unroll
		for (int j = 0; j < E::NSTAT; ++j) u[Q + j] = (double)g.stat[j * g.ps + c];
		double lam[DIM];
		E::template fastest<DIM>(g.pd, u, lam);
		fw.add(g.cflScale, lam);
	}
	const double m = wave_min(fw.dt(g.cflScale));
	int w = (int)((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
	if ((threadIdx.x & 63) == 0 && m < INFINITY) atomic_min_pos(&g.dev->dtmin[g.slot][w & (DT_LANES - 1)], m);
}

// constrainU (euler.cl:697-717) over the interior; ghosts follow by mapping.
template <typename R, template <typename> class EQ>
__global__ void __launch_bounds__(256) constrain_kernel(const GridArgs<R> g) {
	using E = EQ<R>;
	constexpr int Q = E::Q;
	for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < g.ncell; c += (long)gridDim.x * blockDim.x) {
		double u[Q];
#pragma unroll
		for (int j = 0; j < Q; ++j) u[j] = (double)g.U[j * g.ps + c];
		E::constrain(g.pd, u);
#pragma unroll
		for (int j = 0; j < Q; ++j) g.U[j * g.ps + c] = R(u[j]);
	}
}

// ------------------------------------------------------ compensated totals
// Neumaier summation per thread over a fixed cell subset, then a fixed-order
// tree over the block and a second single-block pass over block partials.
struct KSum {
	double s, c;
};
__device__ __forceinline__ KSum ksum_add(KSum a, double x) {
	double t = a.s + x;
	if (fabs(a.s) >= fabs(x)) a.c += (a.s - t) + x;
	else a.c += (x - t) + a.s;
	a.s = t;
	return a;
}
__device__ __forceinline__ KSum ksum_merge(KSum a, KSum b) {
	a = ksum_add(a, b.s);
	a.c += b.c;
	return a;
}

constexpr int TOTALS_BLOCK = 256;

template <typename R>
__global__ void __launch_bounds__(TOTALS_BLOCK) totals_partial_kernel(const R *U, long ps, long ncell, int q, KSum *partial) {
	__shared__ KSum sh[TOTALS_BLOCK];
	for (int j = 0; j < q; ++j) {
		KSum a = {0., 0.};
		for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += (long)gridDim.x * blockDim.x)
			a = ksum_add(a, (double)U[j * ps + c]);
		sh[threadIdx.x] = a;
		__syncthreads();
		for (int w = TOTALS_BLOCK / 2; w > 0; w >>= 1) {
			if ((int)threadIdx.x < w) sh[threadIdx.x] = ksum_merge(sh[threadIdx.x], sh[threadIdx.x + w]);
			__syncthreads();
		}
		if (threadIdx.x == 0) partial[j * gridDim.x + blockIdx.x] = sh[0];
		__syncthreads();
	}
}

[[maybe_unused]] static __global__ void __launch_bounds__(TOTALS_BLOCK) totals_final_kernel(const KSum *partial, int nPartial, int q, double *out) {
	__shared__ KSum sh[TOTALS_BLOCK];
	for (int j = 0; j < q; ++j) {
		KSum a = {0., 0.};
		for (int i = threadIdx.x; i < nPartial; i += blockDim.x) a = ksum_merge(a, partial[j * nPartial + i]);
		sh[threadIdx.x] = a;
		__syncthreads();
		for (int w = TOTALS_BLOCK / 2; w > 0; w >>= 1) {
			if ((int)threadIdx.x < w) sh[threadIdx.x] = ksum_merge(sh[threadIdx.x], sh[threadIdx.x + w]);
			__syncthreads();
		}
		if (threadIdx.x == 0) out[j] = sh[0].s + sh[0].c;
		__syncthreads();
	}
}

// ------------------------------------------------------------ var stats
// calcDisplayVarRangeAndAvgAndStdDev (solverbase.lua:2871-2994) of one
// stored field: min and max over every cell of the ghosted grid (ghost values
// as the boundary fills them: periodic/freeflow copies, mirror flips, fixed
// values), the average and the population standard deviation over the
// interior (the reference zeroes the ghosts for its sums and divides by the
// interior count). One pass (stats_kernel), FP64 compensated sums.
// Derived Euler display variables (euler.lua:240-260) of one cell's cons
// (rho, m, ETotal) in double: W from primFromCons (euler.cl:140-159, P by
// calc_P, euler.cl:63-83), then the variable's formula from euler.cl:1-94.
struct StatsPar {
	double gamma, rhoMin, PMin;
};
__device__ inline double euler_display(const StatsPar &p, int id, const double *U) {
	const double rho = U[0];
	const double inv = 1. / rho;
	const double v[3] = {U[1] * inv, U[2] * inv, U[3] * inv};
	const double mSq = U[1] * U[1] + U[2] * U[2] + U[3] * U[3];
	const double EKinC = rho < p.rhoMin ? 0. : (.5 * mSq / rho);
	const double P = rho < p.rhoMin ? 0. : ((p.gamma - 1.) * (U[4] - EKinC));
	const double vSq = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
	auto Cs = [&]() { return P <= p.PMin ? 0. : rho < p.rhoMin ? (double)INFINITY : sqrt(p.gamma * P / rho); };
	switch (id) {
	case HYDRO_VAR_P: return P;
	case HYDRO_VAR_E_INT_SPEC: return P / (p.gamma - 1.) / rho;
	case HYDRO_VAR_E_KIN_SPEC: return .5 * vSq;
	case HYDRO_VAR_E_TOTAL_SPEC: return U[4] / rho;
	case HYDRO_VAR_E_INT: return P / (p.gamma - 1.);
	case HYDRO_VAR_E_KIN: return rho * (.5 * vSq);
	case HYDRO_VAR_S: return P / pow(rho, p.gamma);
	case HYDRO_VAR_H: return P * (p.gamma / (p.gamma - 1.));
	case HYDRO_VAR_H_SPEC: return P * (p.gamma / (p.gamma - 1.)) / rho;
	case HYDRO_VAR_H_TOTAL: return P + U[4];
	case HYDRO_VAR_H_TOTAL_SPEC: return (P + U[4]) / rho;
	case HYDRO_VAR_CS: return Cs();
	case HYDRO_VAR_MACH: return sqrt(vSq) / Cs();
	case HYDRO_VAR_V_X: return v[0];
	case HYDRO_VAR_V_Y: return v[1];
	default: return v[2];
	}
}

// A double of another lane by DPP; lanes without a source, or of a row that the
// mask leaves out, get `none`.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_double(double v, double none) {
	const int2 p = __builtin_bit_cast(int2, v), n = __builtin_bit_cast(int2, none);
	int2 q;
	q.x = __builtin_amdgcn_update_dpp(n.x, p.x, CTRL, ROWS, 0xF, false);
	q.y = __builtin_amdgcn_update_dpp(n.y, p.y, CTRL, ROWS, 0xF, false);
	return __builtin_bit_cast(double, q);
}

// What a field's statistics are made of: compensated sums of the values, of their
// distances from one of them (d) and of the distances' squares (q), and the range.
struct FieldStats {
	KSum s, d, q;
	double mn, mx;
};
__device__ __forceinline__ FieldStats stats_none() { return {{0., 0.}, {0., 0.}, {0., 0.}, INFINITY, -INFINITY}; }
template <int CTRL, int ROWS>
__device__ __forceinline__ KSum ksum_step(KSum a) {
	return ksum_merge(a, KSum{dpp_double<CTRL, ROWS>(a.s, 0.), dpp_double<CTRL, ROWS>(a.c, 0.)});
}
template <int CTRL, int ROWS>
__device__ __forceinline__ void stats_step(FieldStats &a) {
	a.s = ksum_step<CTRL, ROWS>(a.s);
	a.d = ksum_step<CTRL, ROWS>(a.d);
	a.q = ksum_step<CTRL, ROWS>(a.q);
	a.mn = fmin(a.mn, dpp_double<CTRL, ROWS>(a.mn, a.mn));
	a.mx = fmax(a.mx, dpp_double<CTRL, ROWS>(a.mx, a.mx));
}
// The block's result in every thread's return value (its first use of sh must
// be behind a barrier of the caller's): lanes by DPP, in lane 63, then the waves
// in order.
__device__ __forceinline__ FieldStats stats_block(FieldStats a, FieldStats *sh) {
	stats_step<0x111, 0xF>(a);
	stats_step<0x112, 0xF>(a);
	stats_step<0x114, 0xF>(a);
	stats_step<0x118, 0xF>(a);
	stats_step<0x142, 0xA>(a);
	stats_step<0x143, 0xC>(a);
	if ((threadIdx.x & 63) == 63) sh[threadIdx.x >> 6] = a;
	__syncthreads();
	FieldStats r = sh[0];
	for (int w = 1; w < TOTALS_BLOCK / WAVE; ++w) {
		r.s = ksum_merge(r.s, sh[w].s);
		r.d = ksum_merge(r.d, sh[w].d);
		r.q = ksum_merge(r.q, sh[w].q);
		r.mn = fmin(r.mn, sh[w].mn);
		r.mx = fmax(r.mx, sh[w].mx);
	}
	return r;
}

// The sum of squares about the mean from the sums about another point:
// q - d^2 / n, in twice the precision, since it may cancel by a factor of n.
__device__ __forceinline__ double stats_squares(const FieldStats &a, double n) {
	const double dh = a.d.s + a.d.c, dl = (a.d.s - dh) + a.d.c;
	const double qh = a.q.s + a.q.c, ql = (a.q.s - qh) + a.q.c;
	const double p = dh * dh, pl = fma(dh, dh, -p) + 2. * dh * dl;
	const double mh = p / n, ml = (fma(-mh, n, p) + pl) / n;
	const double v = (qh - mh) + (ql - ml);
	return v < 0. ? 0. : v;
}

// The statistics of a field in one pass: range, average, standard deviation. The
// deviations are taken from the first interior value instead of the average, which
// would need a pass before; their squares are summed with their rounding errors, all
// sums compensated. The interior is one dense run per
// plane; ghosts can only matter to the range, and only where a face is mirrored
// or fixed (ghosts of the others repeat interior values): those are then visited
// on their own. The last block to finish puts the blocks' results together in
// their order, so the result does not depend on which it is, leaves the
// ticket at 0 and writes all four numbers to host memory (pinned) or out.
// A launch of dependent loads and reductions, bound by latency up to some
// 10^6 cells: from call to numbers 256^2 FP64 67 -> 25, 600x400 69 -> 24, 1024^2 84 -> 28 us; a
// field of 256^3 FP32, bound by its read, 215 -> 132 (two passes, each of two launches
// at first).
template <typename R, template <typename> class EQ>
__global__ void __launch_bounds__(TOTALS_BLOCK) stats_kernel(const GridDesc<R> g, int dim, int field, int ghosts,
	double nInterior, FieldStats *partial, double *out, double *host, StatsPar sp)
{
	using E = EQ<R>;
	__shared__ FieldStats sh[2][TOTALS_BLOCK / WAVE];
	__shared__ int last;
	const long ncell = (long)g.n[0] * g.n[1] * g.n[2];
	const long first = (long)blockIdx.x * blockDim.x + threadIdx.x, stride = (long)gridDim.x * blockDim.x;
	FieldStats a = stats_none();
	const bool derived = E::Q == 5 && field >= HYDRO_VAR_P;
	const R *plane = derived ? nullptr : field < E::Q ? g.U[0] + (long)field * g.ps : g.stat + (long)(field - E::Q) * g.ps;
	auto value = [&](long c) {
		if (!derived) return (double)plane[c];
		double U[5];
#pragma unroll
		for (int f = 0; f < 5; ++f) U[f] = (double)g.U[0][f * g.ps + c];
		return euler_display(sp, field, U);
	};
	const double x0 = value(0);
	for (long c = first; c < ncell; c += stride) {
		const double x = value(c), d = x - x0, dd = d * d;
		a.mn = fmin(a.mn, x);
		a.mx = fmax(a.mx, x);
		a.s = ksum_add(a.s, x);
		a.d = ksum_add(a.d, d);
		a.q = ksum_add(a.q, dd);
		a.q.c += fma(d, d, -dd);
	}
	if (ghosts) {
		// ghost planes in z (whole), ghost rows in y of the others (whole), then
		// the 2 + 2 ghosts of every interior row
		const int gx = g.n[0] + 2 * NG, gy = dim > 1 ? g.n[1] + 2 * NG : 1;
		const long rowsZ = dim > 2 ? 2L * NG * gy : 0, rowsY = dim > 1 ? 2L * NG * g.n[2] : 0;
		const long whole = (rowsZ + rowsY) * gx, total = whole + 2L * NG * g.n[1] * g.n[2];
		for (long i = first; i < total; i += stride) {
			int cc[3];
			if (i < whole) {
				const long row = i / gx;
				cc[0] = (int)(i - row * gx) - NG;
				if (row < rowsZ) {
					const int k = (int)(row / gy);
					cc[2] = k < NG ? k - NG : g.n[2] + k - NG;
					cc[1] = (int)(row % gy) - (dim > 1 ? NG : 0);
				} else {
					const long r = row - rowsZ;
					const int j = (int)(r % (2 * NG));
					cc[2] = (int)(r / (2 * NG));
					cc[1] = j < NG ? j - NG : g.n[1] + j - NG;
				}
			} else {
				const long r = (i - whole) / (2 * NG);
				const int j = (int)((i - whole) % (2 * NG));
				cc[0] = j < NG ? j - NG : g.n[0] + j - NG;
				cc[1] = (int)(r % g.n[1]);
				cc[2] = (int)(r / g.n[1]);
			}
			Mapped m[3];
#pragma unroll
			for (int d = 0; d < 3; ++d) {
				if (d < dim) m[d] = map_coord(cc[d], g.n[d], g.bc[2 * d], g.bc[2 * d + 1], 2 * d);
				else { m[d].idx = 0; m[d].mirror = 0; m[d].fixedFace = -1; }
			}
			const long src = ((long)m[2].idx * g.n[1] + m[1].idx) * g.step1 + m[0].idx;
			// axis by axis as the boundary passes run: a fixed face writes its
			// value, a mirror face flips the reflected fields
			auto fieldAt = [&](int f) {
				R v = f < E::Q ? g.U[0][f * g.ps + src] : g.stat[(f - E::Q) * g.ps + src];
#pragma unroll
				for (int d = 0; d < 3; ++d) {
					if (m[d].fixedFace >= 0) v = g.fixedv[m[d].fixedFace][f];
					else if (m[d].mirror && E::reflects(f, d)) v = -v;
				}
				return (double)v;
			};
			double x;
			if (derived) {
				double U[5];
				for (int f = 0; f < 5; ++f) U[f] = fieldAt(f);
				x = euler_display(sp, field, U);
			} else {
				x = fieldAt(field);
			}
			a.mn = fmin(a.mn, x);
			a.mx = fmax(a.mx, x);
		}
	}
	a = stats_block(a, sh[0]);
	if (threadIdx.x == 0) {
		partial[blockIdx.x] = a;
		__threadfence();
		last = atomicAdd(&g.dev->ticket, 1u) == gridDim.x - 1;
	}
	__syncthreads();
	if (!last) return;
	__threadfence();
	a = stats_none();
	for (unsigned i = threadIdx.x; i < gridDim.x; i += blockDim.x) {
		const FieldStats o = partial[i];
		a.s = ksum_merge(a.s, o.s);
		a.d = ksum_merge(a.d, o.d);
		a.q = ksum_merge(a.q, o.q);
		a.mn = fmin(a.mn, o.mn);
		a.mx = fmax(a.mx, o.mx);
	}
	a = stats_block(a, sh[1]);
	if (threadIdx.x != 0) return;
	g.dev->ticket = 0u;
	double *to = host ? host : out;
	to[0] = a.mn;
	to[1] = a.mx;
	to[2] = (a.s.s + a.s.c) / nInterior;
	to[3] = sqrt(stats_squares(a, nInterior) / nInterior);
}

} // namespace hydro
