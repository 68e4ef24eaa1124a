// The launches of 1D steps: whole ones, many to a launch where the grid fits one block
// and one to a launch beyond it; by stages where one face of the two is periodic, and
// one-stage steps of more waves than start at once.
#include <cstdio>
#include <vector>

#include "hip_stub.h"

// A launch's arguments beyond 1 KiB cost a short kernel .4 us (FP32 1D stages). FP64
// was a little more before there were whole steps.
static_assert(sizeof(hydro::StageArgs<float>) <= 1024 && sizeof(hydro::StageArgs<double>) <= 1344, "launch arguments");

#define REQUIRE(x) do { if (!(x)) { std::printf("failed: %s at %d (%s)\n", #x, __LINE__, hydro_last_error()); return 1; } } while (0)

static std::vector<StubLaunch> seen;

int main() {
	stub.stage = [](const StubLaunch &l) { seen.push_back(l); };
	for (int fast = 0; fast < 2; ++fast)
		for (int integ = 0, order = 0; hydro_integrator_table(integ, &order, nullptr, nullptr) == 0; ++integ)
			for (int n : {1, 64, 300, 384, 385, 480, 481, 1000, 20011, 184320, 184321})
				for (int mixed = 0; mixed < 2; ++mixed) {
					hydro_cfg c;
					hydro_cfg_default(&c);
					c.dim = 1;
					c.size[0] = n;
					c.integrator = integ;
					c.fast_math = fast;
					c.boundary[0] = HYDRO_BC_PERIODIC;
					c.boundary[1] = mixed ? HYDRO_BC_FREEFLOW : HYDRO_BC_PERIODIC;
					hydro_solver *h = nullptr;
					REQUIRE(hydro_create(&c, &h) == 0);
					const bool block = n <= (64 - 4 * order) * 8;
					const bool each = !mixed && (order > 1 || n <= 184320);
					seen.clear();
					REQUIRE(hydro_update(h, 1) == 0);
					REQUIRE((int)seen.size() == (each ? 1 : order) && seen[0].steps == (each ? 1 : 0));
					seen.clear();
					REQUIRE(hydro_update(h, 257) == 0);
					if (!mixed && block)
						REQUIRE((int)seen.size() == 1 + (each ? 1 : order) && seen[0].steps == 256 && seen[1].steps == (each ? 1 : 0));
					else
						REQUIRE((int)seen.size() == 257 * (each ? 1 : order) && seen[9].steps == (each ? 1 : 0));
					hydro_destroy(h);
				}
	std::printf("as ruled\n");
	return 0;
}
