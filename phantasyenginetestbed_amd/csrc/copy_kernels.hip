// Copies between pinned host memory and the device, many ranges per launch.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"

namespace phx {
namespace {

constexpr uint32_t kSegment = 16384;  // bytes a block copies at a time: 256 threads, four 16-B words each

// A launch's ranges in segments: range i has segments first[i] to first[i + 1].
struct Ranges {
	const char* src[kCopyRanges];
	char* dst[kCopyRanges];
	uint64_t bytes[kCopyRanges];
	uint32_t first[kCopyRanges + 1];
	uint32_t count;
};

// Bound by the host link, as a copy call is; what it saves is calls: a request's copy took 20 to 45 us of
// the dispatcher and of the copy engine's queue, so 48 requests of 1,024 to 262,144 rays waited for 96 of
// them.
// Blocks: every read over the link, the device's own of its queues' packets included, waits behind those
// in flight (16 KB a block), so they are no more than fill the link; writes need fewer. A device-resident
// request beside the copy of 4 million rays, 48 requests and 1,500 requests took, in ms:
//   blocks to the device, to the host   64, 64   32, 32   32, 16   24, 64   16, 16
//   4,096 device-resident rays           0.95     0.45     0.52     0.38     0.30
//   48 host requests                     3.20     2.97     3.03     3.14     3.50
//   1,500 host requests                  64.7     66.7     65.0     71.7     86.5
__global__ __launch_bounds__(256) void k_copy_ranges(Ranges R)
{
	const uint32_t segments = R.first[R.count];
	for (uint32_t s = blockIdx.x; s < segments; s += gridDim.x) {
		uint32_t lo = 0, hi = R.count;
		while (hi - lo > 1) {
			const uint32_t mid = (lo + hi) >> 1;
			if (R.first[mid] <= s)
				lo = mid;
			else
				hi = mid;
		}
		const uint64_t at = uint64_t(s - R.first[lo]) * kSegment;
		const char* src = R.src[lo] + at;
		char* dst = R.dst[lo] + at;
		const uint32_t bytes = uint32_t(R.bytes[lo] - at < kSegment ? R.bytes[lo] - at : kSegment);
		const uint32_t words = bytes / 16u;
		uint4 w[4];
#pragma unroll
		for (uint32_t k = 0; k < 4u; k++) {
			const uint32_t i = threadIdx.x + k * 256u;
			if (i < words) w[k] = reinterpret_cast<const uint4*>(src)[i];
		}
#pragma unroll
		for (uint32_t k = 0; k < 4u; k++) {
			const uint32_t i = threadIdx.x + k * 256u;
			if (i < words) reinterpret_cast<uint4*>(dst)[i] = w[k];
		}
		const uint32_t tail = words * 16u + threadIdx.x;
		if (tail < bytes) dst[tail] = src[tail];
	}
}

}  // namespace

void* deviceAddress(const void* p, size_t bytes)
{
	if (!p || bytes == 0) return nullptr;
	hipPointerAttribute_t at{};
	if (hipPointerGetAttributes(&at, p) != hipSuccess) {
		(void)hipGetLastError();  // not known to the runtime: pageable
		return nullptr;
	}
	if (at.type != hipMemoryTypeHost || !at.devicePointer) return nullptr;
	// All of it in the allocation of its first byte: between two allocations there may be pageable memory.
	hipDeviceptr_t base = nullptr;
	size_t size = 0;
	if (hipMemGetAddressRange(&base, &size, at.devicePointer) != hipSuccess) {
		(void)hipGetLastError();
		return nullptr;
	}
	const uintptr_t first = reinterpret_cast<uintptr_t>(at.devicePointer), start = reinterpret_cast<uintptr_t>(base);
	if (first < start || first - start > size || bytes > size - (first - start)) return nullptr;
	return first % 16u == 0u ? at.devicePointer : nullptr;
}

hipError_t launchCopies(const CopyRange* ranges, uint32_t count, bool toHost, hipStream_t stream)
{
	const uint64_t most = toHost ? 16u : 32u;
	for (uint32_t at = 0; at < count;) {
		Ranges R{};
		uint64_t segments = 0;
		while (at < count && R.count < kCopyRanges) {
			const uint64_t more = (ranges[at].bytes + kSegment - 1u) / kSegment;
			if (segments + more > 0x7FFFFFFFull) break;
			R.src[R.count] = static_cast<const char*>(ranges[at].src);
			R.dst[R.count] = static_cast<char*>(ranges[at].dst);
			R.bytes[R.count] = ranges[at].bytes;
			R.first[R.count++] = uint32_t(segments);
			segments += more;
			at++;
		}
		R.first[R.count] = uint32_t(segments);
		if (R.count == 0) return hipErrorInvalidValue;
		hipLaunchKernelGGL(k_copy_ranges, dim3(uint32_t(std::min<uint64_t>(std::max<uint64_t>(segments, 1u), most))),
		                   dim3(256), 0, stream, R);
		const hipError_t e = hipGetLastError();
		if (e != hipSuccess) return e;
	}
	return hipSuccess;
}

}  // namespace phx
