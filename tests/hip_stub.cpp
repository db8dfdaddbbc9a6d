// A HIP runtime without a device, for tests of the host code on the CPU:
// loaded with RTLD_GLOBAL before libccf_amd.so, it takes the place of the
// runtime's functions. Memory is host memory (zeroed), copies and fills are
// done at once, kernels are not run. Every launch, copy, pinned allocation
// and synchronisation is written to the file stub_log() names, one a line;
// stub_fail(kernel, n) makes the n-th launch of a kernel from then on fail.
//
// Built and used by test_host_launches.py.
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace
{
std::mutex mu;
std::map<const void*, std::string> names;
std::map<const char*, size_t> pinned;
FILE* out = nullptr;
std::string fail_name;
int fail_at = 0, cus = 256;
thread_local hipError_t last = hipSuccess;
struct Config
{
	dim3 grid, block;
	size_t lds;
	hipStream_t stream;
};
thread_local Config config;

long id(const void* p) { return p ? *(const long*)p : 0; }
void* handle()
{
	static long next = 0;
	std::lock_guard<std::mutex> l(mu);
	return new long(++next);
}
void line(const char* f, ...)
{
	std::lock_guard<std::mutex> l(mu);
	if (!out) return;
	va_list a;
	va_start(a, f);
	std::vfprintf(out, f, a);
	va_end(a);
	std::fflush(out);
}
} // namespace

extern "C" {

void stub_log(const char* path)
{
	std::lock_guard<std::mutex> l(mu);
	if (out) std::fclose(out);
	out = path ? std::fopen(path, "w") : nullptr;
}
void stub_fail(const char* kernel, int n)
{
	fail_name = kernel;
	fail_at = n;
}
void stub_cus(int n) { cus = n; }

void** __hipRegisterFatBinary(const void*) { return (void**)handle(); }
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*)
{
	std::lock_guard<std::mutex> l(mu);
	names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s)
{
	config = {g, b, lds, s};
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s)
{
	*g = config.grid;
	*b = config.block;
	*lds = config.lds;
	*s = config.stream;
	return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t s)
{
	std::string n;
	{
		std::lock_guard<std::mutex> l(mu);
		n = names[f];
	}
	line("launch %s %u %u %u %u stream %ld\n", n.c_str(), g.x, g.y, g.z, b.x, id(s));
	if (fail_at > 0 && n.find(fail_name) != std::string::npos && --fail_at == 0) return last = hipErrorLaunchFailure;
	return hipSuccess;
}
hipError_t hipGetLastError()
{
	const hipError_t e = last;
	last = hipSuccess;
	return e;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipGetDeviceCount(int* n)
{
	*n = 1;
	return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevice(int* d)
{
	*d = 0;
	return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t a, int)
{
	*v = a == hipDeviceAttributeMultiprocessorCount ? cus : (a == hipDeviceAttributeMaxSharedMemoryPerBlock ? 163840 : 0);
	return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t)
{
	*n = 2;
	return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*)
{
	*p = nullptr;
	return hipErrorInvalidSymbol;
}

hipError_t hipMalloc(void** p, size_t n)
{
	*p = std::calloc(1, n);
	return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void* p)
{
	std::free(p);
	return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
	*p = std::calloc(1, n);
	line("pin %zu\n", n);
	std::lock_guard<std::mutex> l(mu);
	pinned[(const char*)*p] = n;
	return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p)
{
	line("unpin\n");
	std::lock_guard<std::mutex> l(mu);
	pinned.erase((const char*)p);
	std::free(p);
	return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
	std::memset(a, 0, sizeof(*a));
	a->type = hipMemoryTypeUnregistered;
	std::lock_guard<std::mutex> l(mu);
	const auto it = pinned.upper_bound((const char*)p);
	if (it != pinned.begin() && (const char*)p < std::prev(it)->first + std::prev(it)->second) a->type = hipMemoryTypeHost;
	return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
	std::memcpy(d, s, n);
	line("copy %zu to %p\n", n, d);
	return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st)
{
	std::memcpy(d, s, n);
	line("copy %zu to %p stream %ld\n", n, d, id(st));
	return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t)
{
	std::memset(d, v, n);
	return hipSuccess;
}

hipError_t hipStreamCreate(hipStream_t* s)
{
	*s = (hipStream_t)handle();
	return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s)
{
	line("sync stream %ld\n", id(s));
	return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
	*e = (hipEvent_t)handle();
	return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
	line("record %ld stream %ld\n", id(e), id(s));
	return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
	*ms = 1;
	return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
	line("wait %ld stream %ld\n", id(e), id(s));
	return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g)
{
	*g = (hipGraph_t)handle();
	return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
	*e = (hipGraphExec_t)handle();
	return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }

} // extern "C"
