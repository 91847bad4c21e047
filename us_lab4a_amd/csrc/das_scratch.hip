// Device scratch of the no-allocation DAS, in a translation unit of its own: GPU
// code is loaded a unit at a time, when something of it is first used.  Beside the
// kernels of das.hip its 256 MiB were loaded with every process's first frame (its
// DAS 107 ms; now 4.7, and the first call that uses the scratch 102).
#include "common.h"

#include <map>
#include <mutex>

namespace mista {

// The tile delays, window tables and per-rx sums of as many tiles as fit.  Every
// call on a GPU shares that GPU's copy (each GPU that the entry point ran on holds
// one until the process ends) and rebuilds what it needs: calls that overlap on
// one GPU race.  In host code `scratch` names a host-side stand-in; kernels get the
// device address from hipGetSymbolAddress.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
std::mutex g_scratch_mu;
std::map<int, unsigned char*> g_scratch_ptr;   // device ordinal -> that GPU's copy of scratch
}  // namespace

unsigned char* noalloc_scratch()
{
	int dev = 0;
	HIP_CHECK(hipGetDevice(&dev));
	std::lock_guard<std::mutex> g(g_scratch_mu);
	auto it = g_scratch_ptr.find(dev);
	if (it != g_scratch_ptr.end()) return it->second;
	void* ptr = nullptr;
	HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
	g_scratch_ptr[dev] = static_cast<unsigned char*>(ptr);
	return static_cast<unsigned char*>(ptr);
}

}  // namespace mista
