// Which kernel a plain solver launches: setting the launch shape that it reports
// changes nothing, more rows select the marching kernel and one row the tile
// kernel where the grid is one of its.
#include <cstdio>
#include <vector>

#include "hip_stub.h"

#define REQUIRE(x) do { if (!(x)) { std::printf("failed: %s at %d (%s)\n", #x, __LINE__, hydro_last_error()); return 1; } } while (0)

static std::vector<StubLaunch> seen;

// the launches of `steps` updates
static std::vector<StubLaunch> update(hydro_solver *h, int steps) {
	seen.clear();
	if (hydro_update(h, steps)) seen.clear();
	return seen;
}

static bool same(const std::vector<StubLaunch> &a, const std::vector<StubLaunch> &b) {
	if (a.empty() || a.size() != b.size()) return false;
	for (size_t i = 0; i < a.size(); ++i)
		if (a[i].tile != b[i].tile || a[i].steps != b[i].steps || a[i].stripsX != b[i].stripsX ||
			(!a[i].tile && (a[i].rows != b[i].rows || a[i].items != b[i].items))) return false;
	return true;
}

int main() {
	stub.stage = [](const StubLaunch &l) { seen.push_back(l); };
	const int sizes[][3] = {{64, 60, 1}, {256, 256, 1}, {500, 380, 1}, {1024, 1024, 1}, {2000, 1500, 1}, {64, 48, 40}, {200, 1, 1}};
	for (auto &n : sizes)
		for (int eqn = 0; eqn < 3; ++eqn) {
			hydro_cfg c;
			hydro_cfg_default(&c);
			c.dim = n[2] > 1 ? 3 : n[1] > 1 ? 2 : 1;
			if (eqn && c.dim == 3) continue;
			c.eqn = eqn;
			c.fast_math = 1;
			c.gravity = 1;
			for (int i = 0; i < 3; ++i) c.size[i] = n[i];
			hydro_solver *h = nullptr;
			REQUIRE(hydro_create(&c, &h) == 0);
			const auto byDefault = update(h, 3);
			int rows = 0, xcd = 0, again = 0;
			REQUIRE(hydro_get_launch(h, &rows, &xcd) == 0);
			REQUIRE(hydro_set_launch(h, rows, xcd) == 0);
			REQUIRE(same(update(h, 3), byDefault));
			if (c.dim == 2) {
				REQUIRE((byDefault[0].tile != 0) == (n[0] <= 256 || (n[0] == 500 && eqn != HYDRO_EQN_GLM_MAXWELL)));
				REQUIRE(hydro_set_launch(h, rows == 4 ? 5 : 4, 0) == 0);
				REQUIRE(!same(update(h, 3), byDefault) && !seen[0].tile);
			}
			REQUIRE(hydro_set_launch(h, rows, xcd) == 0);
			REQUIRE(same(update(h, 3), byDefault));
			REQUIRE(hydro_get_launch(h, &again, nullptr) == 0 && again == rows);
			hydro_destroy(h);
		}
	// a kernel of two waves a SIMD: IEEE, whose division sequences fill more of one, takes
	// five rows in one round where a fast one takes three in waves that run in pairs
	stub.occupancy = 2;
	for (int fast = 0; fast < 2; ++fast) {
		hydro_cfg c;
		hydro_cfg_default(&c);
		c.dim = 2;
		c.size[0] = 640;
		c.size[1] = 480;
		c.plm = HYDRO_PLM_ATHENA;
		c.fast_math = fast;
		hydro_solver *h = nullptr;
		int rows = 0;
		REQUIRE(hydro_create(&c, &h) == 0 && hydro_get_launch(h, &rows, nullptr) == 0);
		REQUIRE(rows == (fast ? 3 : 5));
		hydro_destroy(h);
	}
	std::printf("as reported\n");
	return 0;
}
