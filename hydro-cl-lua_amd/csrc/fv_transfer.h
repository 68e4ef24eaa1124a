// fv_transfer.h — host <-> device transfers of the plain and batched solvers:
// the reference's ghosted cons_t buffer (cells, caller's memory) against the
// planes of the interior on the device.
//
// The buffer goes through pinned slots, chunk by chunk: a kernel converts between
// cells and planes while it crosses the bus (give_cells_kernel,
// take_cells_kernel, fv_aux.h), and the host only copies whole chunks between the
// caller's memory and the slots, on up to 8 threads with two slots each, so that
// the copy of one chunk overlaps the bus time of others. What bounds a large
// transfer is the host's copy (first touches of the caller's pages included).
// Before, the host packed and unpacked the cells itself beside pageable copies of
// all planes: down 256^2 FP64 .47 -> .19, 1024^2 13 -> 1.6, 256^3 FP32 107 -> 9.8;
// up 1024^2 FP64 10.4 -> 1.3, 256^3 FP32 84 -> 10.6 ms (42 GB/s of the buffer).
#pragma once

#include <atomic>
#include <condition_variable>
#include <mutex>

#include "fv_host.h"

namespace hydro {

// Pinned slots shared by every solver and batch of the process: at most
// MAX_SLOTS, made as they are needed and freed with the last handle. A transfer's
// threads keep theirs from chunk to chunk until another's wait for one (wanted), so
// that a small transfer beside a large one waits for a chunk of it and not for all.
class PinnedSlots {
public:
	static constexpr size_t SLOT = (size_t)2 << 20;
	static constexpr int MAX_SLOTS = 16;

	void add_handle() {
		std::lock_guard<std::mutex> lock(mu);
		++handles;
	}
	void drop_handle() {
		std::lock_guard<std::mutex> lock(mu);
		if (--handles > 0) return;
		for (char *p : idle) ignore(hipHostFree(p));
		made -= (int)idle.size();
		idle.clear();
	}
	// A slot, in the order of the calls; nullptr if there are none and none can be
	// made. The caller holds none itself, so that each that is taken comes back.
	char *take() {
		std::unique_lock<std::mutex> lock(mu);
		const long turn = last++;
		++waiting;
		char *p = nullptr;
		freed.wait(lock, [&] { return turn == turns && ((p = get()) || made == 0); });
		--waiting;
		++turns;
		lock.unlock();
		freed.notify_all();
		return p;
	}
	// Up to `want` slots that can be had at once, if nobody waits for one.
	int try_take(int want, char **out) {
		std::lock_guard<std::mutex> lock(mu);
		int n = 0;
		while (n < want && !waiting.load() && (out[n] = get())) ++n;
		return n;
	}
	bool wanted() const { return waiting.load() > 0; }
	void give(char *const *slots, int n) {
		{
			std::lock_guard<std::mutex> lock(mu);
			for (int i = 0; i < n; ++i)
				if (slots[i]) idle.push_back(slots[i]);
		}
		freed.notify_all();
	}

private:
	char *get() {
		if (!idle.empty()) {
			char *p = idle.back();
			idle.pop_back();
			return p;
		}
		void *p = nullptr;
		if (made >= MAX_SLOTS) return nullptr;
		if (hipHostMalloc(&p, SLOT, hipHostMallocPortable) != hipSuccess || !p) {
			(void)hipGetLastError();
			return nullptr;
		}
		++made;
		return (char *)p;
	}

	std::mutex mu;
	std::condition_variable freed;
	std::vector<char *> idle;
	int made = 0, handles = 0;
	long last = 0, turns = 0;            // of take: the next to come, the one whose turn it is
	std::atomic<int> waiting{0};
};

inline PinnedSlots &pinned_slots() {
	static PinnedSlots *p = new PinnedSlots();   // outlives every handle
	return *p;
}

// Below this the packed form (pageable copies of the planes) is as fast: 12 KB
// take 25 us up and 35 down in it, 480 KB 98 and 170 against 43 and 59 through the
// slots, most of them one launch and one event.
static constexpr size_t CHUNKED_MIN = (size_t)96 << 10;

template <typename R>
static int upload_packed(Grid &g, const void *U, hipStream_t s) {
	std::vector<R> planes((size_t)g.Q * g.ps), stat((size_t)g.NSTAT * g.ps);
	pack_interior<R>(g, (const R *)U, planes.data(), stat.data());
	HIPCHECK(hipMemcpyAsync(g.U[0], planes.data(), planes.size() * sizeof(R), hipMemcpyHostToDevice, s));
	if (g.NSTAT) HIPCHECK(hipMemcpyAsync(g.stat, stat.data(), stat.size() * sizeof(R), hipMemcpyHostToDevice, s));
	HIPCHECK(hipStreamSynchronize(s));
	g.dtValid = 0;
	return 0;
}

template <typename R>
static int download_packed(const Grid &g, void *U, hipStream_t s) {
	std::vector<R> planes((size_t)g.Q * g.ps), stat((size_t)g.NSTAT * g.ps);
	HIPCHECK(hipMemcpyAsync(planes.data(), g.U[0], planes.size() * sizeof(R), hipMemcpyDeviceToHost, s));
	if (g.NSTAT) HIPCHECK(hipMemcpyAsync(stat.data(), g.stat, stat.size() * sizeof(R), hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	unpack_with_ghosts<R>(g, planes.data(), stat.data(), (R *)U);
	return 0;
}


// g.ePot from the interior cells of an uploaded buffer
template <typename R>
static void keep_ePot(Grid &g, const R *aos) {
	const int dim = g.dim, nx = g.n[0];
	const long gx = nx + 2 * NG, gy = dim > 1 ? g.n[1] + 2 * NG : 1;
	g.ePot.assign(g.ncell, 0.);
	double *ePot = g.ePot.data();
	parallel_ranges((long)g.n[1] * g.n[2], 64, [&](long r0, long r1) {
		for (long row = r0; row < r1; ++row) {
			const long j = row % g.n[1] + (dim > 1 ? NG : 0), k = row / g.n[1] + (dim > 2 ? NG : 0);
			const R *u = aos + (size_t)(NG + gx * (j + gy * k)) * g.S;
			for (int i = 0; i < nx; ++i) ePot[(size_t)nx * row + i] = (double)u[(size_t)i * g.S + 5];
		}
	});
}

// g.ePot into every cell of a downloaded buffer, ghosts as the other fields'
template <typename R>
static void put_ePot(const Grid &g, R *aos) {
	int gs[3];
	for (int i = 0; i < 3; ++i) gs[i] = i < g.dim ? g.n[i] + 2 * NG : 1;
	const hydro_cfg &c = g.cfg;
	parallel_ranges((long)gs[1] * gs[2], 64, [&](long r0, long r1) {
		for (long row = r0; row < r1; ++row) {
			const int at[3] = {0, (int)(row % gs[1]), (int)(row / gs[1])};
			HostMap m[3] = {{0, 0, -1}, {0, 0, -1}, {0, 0, -1}};
			for (int a = 1; a < g.dim; ++a)
				m[a] = host_map(at[a] - NG, g.n[a], c.boundary[2 * a], c.boundary[2 * a + 1], 2 * a);
			const double *src = g.ePot.data() + (size_t)g.n[0] * (m[1].idx + (size_t)g.n[1] * m[2].idx);
			R *u = aos + (size_t)row * gs[0] * g.S + 5;
			for (int i = 0; i < gs[0]; ++i, u += g.S) {
				m[0] = host_map(i - NG, g.n[0], c.boundary[0], c.boundary[1], 0);
				R v = R(src[m[0].idx]);
				for (int a = 0; a < g.dim; ++a)
					if (m[a].fixedFace >= 0) v = R(c.boundary_fixed[m[a].fixedFace][5]);
				*u = v;
			}
		}
	});
}

template <typename R>
static CellBuffer<R> cell_buffer(const Grid &g) {
	CellBuffer<R> b;
	std::memset(&b, 0, sizeof b);
	b.U = (R *)g.U[0];
	b.stat = (R *)g.stat;
	b.ps = g.ps;
	b.dim = g.dim;
	b.q = g.Q;
	b.nstat = g.NSTAT;
	b.S = g.S;
	for (int i = 0; i < 3; ++i) b.n[i] = g.n[i];
	for (int f = 0; f < 6; ++f) {
		b.bc[f] = g.cfg.boundary[f];
		for (int j = 0; j < g.S; ++j) b.fixedv[f][j] = R(g.cfg.boundary_fixed[f][j]);
	}
	const bool glm = g.cfg.eqn == HYDRO_EQN_GLM_MAXWELL;
	b.vec1 = glm ? 0 : 1;
	b.vec2 = glm ? 3 : -1;
	return b;
}

// Moves the ghosted buffer U (host) up to or down from g's planes through the
// slots, on up to 8 threads that hold up to two each. flags (up): what take_cells
// found. Returns 1 if no slot could be had (nothing was moved).
template <typename R, bool UP>
static int move_cells(const Grid &g, R *U, hipStream_t s, int *flags) {
	const size_t cellBytes = (size_t)g.S * sizeof(R);
	const long total = (long)ghosted_cells(g);
	const size_t bytes = (size_t)total * cellBytes;
	constexpr size_t FLAG_BYTES = 64;        // at a slot's end
	const long maxCells = (long)((PinnedSlots::SLOT - FLAG_BYTES) / cellBytes) / CELLS_BLOCK * CELLS_BLOCK;
	const long hw = std::max(1L, (long)std::thread::hardware_concurrency());
	const long threads = std::max(1L, std::min({8L, hw, (long)(bytes >> 20)}));
	// two chunks a thread at least, a slot's worth at most
	long cells = (total + 2 * threads - 1) / (2 * threads);
	cells = std::min(maxCells, (cells + CELLS_BLOCK - 1) / CELLS_BLOCK * CELLS_BLOCK);
	const long chunks = (total + cells - 1) / cells;
	const long workers = std::min(threads, (chunks + 1) / 2);
	int device = 0;
	hipError_t first = hipGetDevice(&device);
	std::atomic<long> next{0};
	std::atomic<int> err{(int)first}, past{0}, outOfPlane{0};
	const CellBuffer<R> shape = cell_buffer<R>(g);
	// two of each thread; nullptr where there was none to be had, or it was given back
	char *slots[PinnedSlots::MAX_SLOTS] = {};
	static_assert(PinnedSlots::MAX_SLOTS >= 2 * 8, "of eight threads");
	pinned_slots().try_take((int)std::min(2 * workers, chunks), slots);
	auto work = [&](long w, bool ownThread) {
		auto ok = [&](hipError_t e) {
			int none = hipSuccess;
			if (e != hipSuccess) err.compare_exchange_strong(none, (int)e);
			return e == hipSuccess;
		};
		if (ownThread && !ok(hipSetDevice(device))) return;
		struct Held {
			char *&slot;
			hipEvent_t ev;
			long at;                // the chunk the slot holds (down) or last sent (up), -1 none
			int *flag_words() const { return (int *)(slot + PinnedSlots::SLOT - FLAG_BYTES); }
		} held[2] = {{slots[2 * w], nullptr, -1}, {slots[2 * w + 1], nullptr, -1}};
		auto drain = [&](Held &h) {      // the slot's kernel has ended; down: its cells go to the caller
			if (h.at < 0) return;
			if (ok(hipEventSynchronize(h.ev))) {
				if (UP) {
					if (h.flag_words()[0]) past = 1;
					if (h.flag_words()[1]) outOfPlane = 1;
				} else {
					const long c0 = h.at * cells, n = std::min(cells, total - c0);
					std::memcpy((char *)U + (size_t)c0 * cellBytes, h.slot, (size_t)n * cellBytes);
				}
			}
			h.at = -1;
		};
		int i = 0;
		while (err.load() == hipSuccess && next.load() < chunks) {
			drain(held[i]);
			if (held[i].slot && pinned_slots().wanted()) {
				pinned_slots().give(&held[i].slot, 1);
				held[i].slot = nullptr;
			}
			if (!held[i].slot) pinned_slots().try_take(1, &held[i].slot);
			if (!held[i].slot && held[1 - i].slot) {
				i = 1 - i;
				drain(held[i]);
			}
			if (!held[i].slot) held[i].slot = pinned_slots().take();
			if (!held[i].slot) break;
			const long c = next.fetch_add(1);
			if (c >= chunks) break;
			Held &h = held[i];
			if (!h.ev && !ok(hipEventCreateWithFlags(&h.ev, hipEventDisableTiming))) break;
			CellBuffer<R> b = shape;
			b.first = c * cells;
			b.count = std::min(cells, total - b.first);
			b.cells = (R *)h.slot;
			b.flags = h.flag_words();
			b.flags[0] = b.flags[1] = 0;
			if (UP) std::memcpy(b.cells, (const char *)U + (size_t)b.first * cellBytes, (size_t)b.count * cellBytes);
			if (!ok(UP ? launch_take_cells<R>(b, s) : launch_give_cells<R>(b, s))) break;
			if (!ok(hipEventRecord(h.ev, s))) {
				ok(hipStreamSynchronize(s));     // the slot is still read or written
				break;
			}
			h.at = c;
			i = 1 - i;
		}
		drain(held[i]);
		drain(held[1 - i]);
		for (Held &h : held)
			if (h.ev) ignore(hipEventDestroy(h.ev));
		// now, and not when all have ended: another of these threads may wait for one
		pinned_slots().give(slots + 2 * w, 2);
		slots[2 * w] = slots[2 * w + 1] = nullptr;
	};
	std::vector<std::thread> th;
	th.reserve((size_t)workers);
	for (long w = 1; w < workers; ++w) {
		try {
			th.emplace_back(work, w, true);
		} catch (const std::system_error &) {
			break;      // the chunks go to the threads there are
		}
	}
	work(0, false);
	for (auto &t : th) t.join();
	pinned_slots().give(slots, PinnedSlots::MAX_SLOTS);      // of threads that could not be made
	if (err.load() != hipSuccess) return fail("transfer of the cons_t buffer: %s", hipGetErrorString((hipError_t)err.load()));
	if (next.load() < chunks) return 1;      // nobody got a slot
	if (flags) {
		flags[0] = past.load();
		flags[1] = outOfPlane.load();
	}
	return 0;
}

template <typename R>
static int grid_upload_t(Grid &g, const void *U, size_t bytes, hipStream_t s) {
	if (bytes < CHUNKED_MIN) return upload_packed<R>(g, U, s);
	int flags[2] = {0, 0};
	const int rc = move_cells<R, true>(g, (R *)const_cast<void *>(U), s, flags);
	if (rc > 0) return upload_packed<R>(g, U, s);
	if (rc < 0) return rc;
	const bool euler = g.cfg.eqn == HYDRO_EQN_EULER;
	// as pack_interior: out-of-plane momenta that are zero everywhere stay so;
	// ePot is kept on the host where any is not 0
	g.nvel = euler && g.dim < 3 && !flags[1] ? g.dim : 3;
	g.ePot.clear();
	if (euler && flags[0]) keep_ePot<R>(g, (const R *)U);
	g.dtValid = 0;
	return 0;
}

template <typename R>
static int grid_download_t(const Grid &g, void *U, size_t bytes, hipStream_t s) {
	if (bytes < CHUNKED_MIN) return download_packed<R>(g, U, s);
	const int rc = move_cells<R, false>(g, (R *)U, s, nullptr);
	if (rc > 0) return download_packed<R>(g, U, s);
	if (rc == 0 && !g.ePot.empty()) put_ePot<R>(g, (R *)U);
	return rc;
}

static int grid_upload(Grid &g, const void *U, size_t bytes, hipStream_t s) {
	if (!U) return fail("NULL argument");
	size_t need = ghosted_cells(g) * g.S * g.elem;
	if (bytes != need) return fail("upload size %zu != %zu (numCells * numStates * sizeof(real))", bytes, need);
	const int rc = g.elem == 8 ? grid_upload_t<double>(g, U, bytes, s) : grid_upload_t<float>(g, U, bytes, s);
	return rc ? rc : clear_past_nvel(g, s);
}

static int grid_download(const Grid &g, void *U, size_t bytes, hipStream_t s) {
	if (!U) return fail("NULL argument");
	size_t need = ghosted_cells(g) * g.S * g.elem;
	if (bytes != need) return fail("download size %zu != %zu (numCells * numStates * sizeof(real))", bytes, need);
	return g.elem == 8 ? grid_download_t<double>(g, U, bytes, s) : grid_download_t<float>(g, U, bytes, s);
}

} // namespace hydro
