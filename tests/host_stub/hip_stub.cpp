// A HIP runtime of host memory for CPU tests of the host code: device memory is
// malloc'ed, copies and fills run in the call that asks for them, kernels do
// nothing but what the hooks of hip_stub.h do.
#include "hip_stub.h"

#include <cstdlib>
#include <cstring>

using namespace hydro;

StubHooks stub;

extern "C" {
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = std::calloc(n, 1); return *p ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
	if (n >= 1 << 20 && --stub.hostBlocks < 0) return hipErrorOutOfMemory;
	return hipMalloc(p, n);
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
	std::memcpy(d, s, n);
	return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)std::malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { std::free(s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)std::malloc(1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) { std::free(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t e) { return stub.query ? stub.query(e) : hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { *ms = 0; return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipErrorNotSupported; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipErrorNotSupported; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipErrorNotSupported; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipErrorNotSupported; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
}

namespace hydro {
hipError_t launch_reset_slots(DevScalars *, int, hipStream_t) { return hipSuccess; }
hipError_t launch_fold_slot(DevScalars *, int, hipStream_t) { return hipSuccess; }

#define STUB_LAUNCHES(R) \
	template <> hipError_t launch_stage<R>(const StageKey &, const StageArgs<R> &a, dim3 grid, dim3, hipStream_t) { \
		if (grid.x == 0) stage_occupancy = stub.occupancy; \
		else if (stub.stage) stub.stage({a.tile, a.steps, a.g.stripsX, a.g.rowsPerWave, a.g.nItems}); \
		return hipSuccess; } \
	template <> hipError_t launch_dt<R>(int, int, int, const GridArgs<R> &, hipStream_t) { return hipSuccess; } \
	template <> hipError_t launch_constrain<R>(int, int, const GridArgs<R> &, hipStream_t) { return hipSuccess; } \
	template <> hipError_t launch_nonfinite<R>(const R *, const R *, long, long, int, int, unsigned *, hipStream_t) { \
		return hipSuccess; } \
	template <> hipError_t launch_totals<R>(const R *, long, long, int, KSum *, int, double *, hipStream_t) { \
		return hipSuccess; } \
	template <> hipError_t launch_stats<R>(int, int, const GridDesc<R> &, int, KSum *, int, double, double *, double *, \
		const double *, hipStream_t) { return hipSuccess; } \
	template <> hipError_t launch_give_cells<R>(const CellBuffer<R> &b, hipStream_t) { \
		if (stub.give) stub.give(b.n[0]); return hipSuccess; } \
	template <> hipError_t launch_take_cells<R>(const CellBuffer<R> &, hipStream_t) { return hipSuccess; }
STUB_LAUNCHES(double)
STUB_LAUNCHES(float)
} // namespace hydro
