// What a CPU test puts in the place of the device (hip_stub.cpp).
#pragma once

#include <hip/hip_runtime.h>

#include <functional>

#include "../../hydro-cl-lua_amd/csrc/fv_aux.h"
#include "../../hydro-cl-lua_amd/csrc/fv_launch.h"

// what a stage or step launch was asked for
struct StubLaunch {
	int tile, steps, stripsX, rows;
	long items;
};

struct StubHooks {
	int occupancy = 4;                               // blocks of any kernel that a compute unit holds
	std::function<void(const StubLaunch &)> stage;   // launch_stage
	std::function<hipError_t(hipEvent_t)> query;     // hipEventQuery; unset: every event has happened
	int hostBlocks = 1 << 30;                        // large blocks of pinned memory that can still be had
	std::function<void(int)> give;                   // a chunk of a download is launched (the grid's first size)
};
extern StubHooks stub;
