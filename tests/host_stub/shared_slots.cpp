// While one thread downloads a large state, chunk by chunk and slowly, another asks
// a second solver for statistics and a small download: both are there before the
// large one has ended, whose bytes, and every other's, arrive.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

#include "hip_stub.h"

#define REQUIRE(x) do { if (!(x)) { std::printf("failed: %s (%s)\n", #x, hydro_last_error()); return 1; } } while (0)

static hydro_solver *solver(int nx, int ny, std::vector<double> &U) {
	hydro_cfg c;
	hydro_cfg_default(&c);
	c.dim = 2;
	c.size[0] = nx;
	c.size[1] = ny;
	hydro_solver *h = nullptr;
	if (hydro_create(&c, &h)) return nullptr;
	U.assign(hydro_num_cells(h) * 6, 0.);
	return h;
}

int main() {
	std::vector<double> big, small, third;
	hydro_solver *a = solver(1200, 1000, big), *b = solver(64, 60, small), *c = solver(640, 500, third);
	REQUIRE(a && b && c);
	std::atomic<int> launched{0};
	std::atomic<bool> over{false};
	stub.give = [&](int nx) {
		if (nx != 1200) return;
		++launched;
		std::this_thread::sleep_for(std::chrono::milliseconds(60));
	};
	int rcA = -1;
	std::thread large([&] {
		rcA = hydro_download_U(a, big.data(), big.size() * sizeof(double));
		over = true;
	});
	while (!launched) std::this_thread::yield();
	std::this_thread::sleep_for(std::chrono::milliseconds(5));      // the others' slots are taken as well
	double out[4];
	REQUIRE(hydro_var_stats(b, 0, out) == 0);
	const bool statsWaited = over;
	REQUIRE(hydro_download_U(b, small.data(), small.size() * sizeof(double)) == 0);
	const bool smallWaited = over;
	REQUIRE(hydro_download_U(c, third.data(), third.size() * sizeof(double)) == 0);
	large.join();
	REQUIRE(rcA == 0);
	REQUIRE(!statsWaited);
	REQUIRE(!smallWaited);
	// many at once, more threads than slots: every one ends; also with three slots in
	// all (the others' memory cannot be had), and with none
	hydro_destroy(a);
	hydro_destroy(b);
	hydro_destroy(c);
	stub.give = nullptr;
	for (int blocks : {1 << 30, 3, 0}) {
		stub.hostBlocks = blocks;
		std::vector<double> U0;
		hydro_solver *keep = solver(16, 16, U0);     // so that the slots are freed at the end, and not between
		std::vector<std::thread> th;
		std::atomic<int> bad{0};
		for (int k = 0; k < 24; ++k)
			th.emplace_back([&, k] {
				std::vector<double> U;
				double four[4];
				hydro_solver *h = solver(300 + k, 400, U);
				for (int i = 0; h && i < 5; ++i)
					if (hydro_upload_U(h, U.data(), U.size() * sizeof(double)) || hydro_var_stats(h, 0, four) ||
						hydro_download_U(h, U.data(), U.size() * sizeof(double))) ++bad;
				if (!h) ++bad;
				hydro_destroy(h);
			});
		for (auto &t : th) t.join();
		hydro_destroy(keep);
		REQUIRE(bad == 0);
	}
	std::printf("shared\n");
	return 0;
}
