// A HIP runtime without a device, for tests of the library's host code on the CPU: linked with the
// library's own objects in place of the real runtime. Device memory cannot be touched by the CPU (a
// host access ends the process, as it may where device memory is not mapped); copies and fills work on
// it. Kernels do not run: launches, event waits, copies and allocations are written to a log that the
// test reads with fake_log.
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>
#include <unistd.h>

#include <atomic>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {

struct Range {
	char* shadow;  // where copies reach the memory (host memory: the memory itself)
	size_t size;
	bool host;
};

std::mutex mu;
std::map<char*, Range> ranges;
std::map<const void*, std::string> kernels;
std::map<const void*, void*> variables;
std::string text;
uintptr_t nextHandle = 1;
std::atomic<bool> held{false};  // copies to the device wait

template <class... A>
void say(const char* format, A... a)
{
	char line[512];
	std::snprintf(line, sizeof(line), format, a...);
	std::lock_guard<std::mutex> g(mu);
	text += line;
	text += '\n';
}

const std::pair<char* const, Range>* find(const void* p)
{
	char* c = static_cast<char*>(const_cast<void*>(p));
	auto it = ranges.upper_bound(c);
	if (it == ranges.begin()) return nullptr;
	--it;
	return c < it->first + it->second.size ? &*it : nullptr;
}

char* reach(const void* p)
{
	std::lock_guard<std::mutex> g(mu);
	char* c = static_cast<char*>(const_cast<void*>(p));
	const auto* r = find(p);
	return r ? r->second.shadow + (c - r->first) : c;
}

template <class H>
hipError_t handle(H* out)
{
	std::lock_guard<std::mutex> g(mu);
	*out = reinterpret_cast<H>(nextHandle++);
	return hipSuccess;
}

hipError_t deviceMemory(void** p, size_t size)
{
	const size_t page = 4096, n = (size + page - 1) / page * page;
	const int fd = memfd_create("device", 0);
	if (fd < 0 || ftruncate(fd, off_t(n)) != 0) return hipErrorOutOfMemory;
	void* shadow = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_SHARED, fd, 0);
	*p = mmap(nullptr, n, PROT_NONE, MAP_SHARED, fd, 0);
	close(fd);
	if (shadow == MAP_FAILED || *p == MAP_FAILED) return hipErrorOutOfMemory;
	std::lock_guard<std::mutex> g(mu);
	ranges[static_cast<char*>(*p)] = Range{static_cast<char*>(shadow), n, false};
	return hipSuccess;
}

template <class T>
T arg(void** args, int i)
{
	T v;
	std::memcpy(&v, args[i], sizeof(v));
	return v;
}

struct Configuration {
	dim3 grid, block;
	size_t lds;
	hipStream_t stream;
};
thread_local Configuration configuration;

}  // namespace

extern "C" {

// Takes what was logged so far: its length, and up to `room` bytes of it.
size_t fake_log(char* out, size_t room)
{
	std::lock_guard<std::mutex> g(mu);
	const size_t n = text.size();
	std::memcpy(out, text.data(), n < room ? n : room);
	text.clear();
	return n;
}

// Holds copies to the device up, as a stream that is busy does copies from pageable memory.
void fake_hold(int on) { held = on != 0; }

void** __hipRegisterFatBinary(const void*)
{
	static void* module;
	return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*)
{
	kernels[f] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int)
{
	void* p = nullptr;
	if (deviceMemory(&p, size) == hipSuccess) variables[var] = p;
}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t stream)
{
	configuration = {grid, block, lds, stream};
	return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* stream)
{
	*grid = configuration.grid, *block = configuration.block;
	*lds = configuration.lds, *stream = configuration.stream;
	return hipSuccess;
}

hipError_t hipLaunchKernel(const void* f, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t stream)
{
	const std::string name = kernels.count(f) ? kernels[f] : "?";
	char more[128] = "";
	if (name.find("k_trace_batches") != std::string::npos)
		std::snprintf(more, sizeof(more), " rays=%u window=%u refill=%u", arg<uint32_t>(args, 3),
		              arg<uint32_t>(args, 4), arg<uint32_t>(args, 5));
	else if (name.find("k_quad") != std::string::npos)
		std::snprintf(more, sizeof(more), " rays=%u window=%u refill=%u", arg<uint32_t>(args, 5),
		              arg<uint32_t>(args, 6), arg<uint32_t>(args, 7));
	say("kernel %s grid=%u block=%u lds=%zu stream=%p%s", name.c_str(), grid.x, block.x, lds,
	    static_cast<void*>(stream), more);
	return hipSuccess;
}

hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
	std::memset(p, 0, sizeof(*p));
	p->multiProcessorCount = 256;
	std::strcpy(p->gcnArchName, "gfx950");
	return hipSuccess;
}
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
hipError_t hipMemGetInfo(size_t* freeB, size_t* total)
{
	*freeB = *total = size_t(288) << 30;
	return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetLastError() { return hipSuccess; }

hipError_t hipMalloc(void** p, size_t size)
{
	const hipError_t e = deviceMemory(p, size ? size : 1);
	if (e == hipSuccess) say("malloc %zu", size);
	return e;
}
hipError_t hipFree(void* p)
{
	if (!p) return hipSuccess;
	std::lock_guard<std::mutex> g(mu);
	const auto it = ranges.find(static_cast<char*>(p));
	if (it == ranges.end() || it->second.host) return hipErrorInvalidValue;
	munmap(it->second.shadow, it->second.size);
	munmap(p, it->second.size);
	ranges.erase(it);
	return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t size, unsigned)
{
	const size_t n = (size + 4095) / 4096 * 4096;
	*p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
	if (*p == MAP_FAILED) return hipErrorOutOfMemory;
	std::lock_guard<std::mutex> g(mu);
	ranges[static_cast<char*>(*p)] = Range{static_cast<char*>(*p), n, true};
	return hipSuccess;
}
// Makes [p, p + size) known as a pinned allocation of its own (memory of the test's).
void fake_pin(void* p, size_t size)
{
	std::lock_guard<std::mutex> g(mu);
	ranges[static_cast<char*>(p)] = Range{static_cast<char*>(p), size, true};
}
hipError_t hipHostFree(void* p)
{
	if (!p) return hipSuccess;
	std::lock_guard<std::mutex> g(mu);
	const auto it = ranges.find(static_cast<char*>(p));
	if (it == ranges.end() || !it->second.host) return hipErrorInvalidValue;
	munmap(p, it->second.size);
	ranges.erase(it);
	return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
	std::lock_guard<std::mutex> g(mu);
	const auto* r = find(p);
	if (!r) return hipErrorInvalidValue;
	std::memset(a, 0, sizeof(*a));
	a->type = r->second.host ? hipMemoryTypeHost : hipMemoryTypeDevice;
	a->devicePointer = const_cast<void*>(p);
	a->hostPointer = r->second.host ? const_cast<void*>(p) : nullptr;
	return hipSuccess;
}
hipError_t hipMemGetAddressRange(hipDeviceptr_t* base, size_t* size, hipDeviceptr_t p)
{
	std::lock_guard<std::mutex> g(mu);
	const auto* r = find(p);
	if (!r) return hipErrorNotFound;
	*base = r->first;
	*size = r->second.size;
	return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* symbol)
{
	*p = variables.count(symbol) ? variables[symbol] : nullptr;
	return *p ? hipSuccess : hipErrorInvalidSymbol;
}

hipError_t hipMemcpy(void* dst, const void* src, size_t n, hipMemcpyKind)
{
	std::memmove(reach(dst), reach(src), n);
	return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t stream)
{
	say("copy %zu kind=%d stream=%p", n, int(kind), static_cast<void*>(stream));
	while (held && kind == hipMemcpyHostToDevice) usleep(1000);
	return hipMemcpy(dst, src, n, kind);
}
hipError_t hipMemset(void* dst, int v, size_t n)
{
	std::memset(reach(dst), v, n);
	return hipSuccess;
}
hipError_t hipMemsetAsync(void* dst, int v, size_t n, hipStream_t) { return hipMemset(dst, v, n); }

hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
	say("wait stream=%p event=%p", static_cast<void*>(s), static_cast<void*>(e));
	return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t* g, hipGraph_t, hipGraphNode_t*, char*, size_t)
{
	return handle(g);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
	say("record stream=%p event=%p", static_cast<void*>(s), static_cast<void*>(e));
	return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
	*ms = 1.0f;
	return hipSuccess;
}

}  // extern "C"
