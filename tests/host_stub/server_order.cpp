// A pool's older chunk ends between the query of its own event, which finds it
// running, and the query of the younger one's, which finds it ended. The requests
// still complete in the order their chunks were launched: one that the older chunk
// uploaded and the younger copied out can be fetched, and the server ticked on.
#include <cstdio>
#include <vector>

#include "hip_stub.h"

#define REQUIRE(x) do { if (!(x)) { std::printf("failed: %s (%s)\n", #x, hydro_last_error()); return 1; } } while (0)

int main() {
	for (int late = 1; late <= 6; ++late) {
		hydro_server *s = nullptr;
		REQUIRE(hydro_server_create((size_t)8 << 20, 20, &s) == 0);
		hydro_cfg c;
		hydro_cfg_default(&c);
		c.dim = 1;
		c.size[0] = 64;
		int order = 0;
		for (c.integrator = 0; order != 2; ++c.integrator)
			REQUIRE(hydro_integrator_table(c.integrator, &order, nullptr, nullptr) == 0);
		--c.integrator;
		std::vector<double> U((64 + 4) * 6, 1.);
		// the `late` first queries find their event still to come
		int queries = 0;
		stub.query = [&](hipEvent_t) { return ++queries <= late ? hipErrorNotReady : hipSuccess; };
		std::vector<long long> ids(3);
		const int steps[3] = {30, 20, 50};      // in two chunks, one and three
		for (int i = 0; i < 3; ++i)
			REQUIRE(hydro_server_submit(s, &c, U.data(), U.size() * sizeof(double), steps[i], &ids[i]) == 0);
		int fetched = 0;
		for (int tick = 0; tick < 20; ++tick) {
			int n = 0;
			REQUIRE(hydro_server_tick(s, &n) == 0);
			long long done[3];
			int have = 0;
			REQUIRE(hydro_server_poll(s, done, 3, &have) == 0);
			for (int i = 0; i < have; ++i) {
				double t = 0;
				int status = 0;
				REQUIRE(hydro_server_result(s, done[i], U.data(), U.size() * sizeof(double), &t, &status) == 0);
				++fetched;
			}
		}
		hydro_server_info info;
		REQUIRE(hydro_server_info_get(s, &info) == 0);
		REQUIRE(fetched == 3 && info.resident == 0 && info.finished == 0 && info.bytes_in_use == 0);
		REQUIRE(hydro_server_destroy(s) == 0);
	}
	std::printf("in order\n");
	return 0;
}
