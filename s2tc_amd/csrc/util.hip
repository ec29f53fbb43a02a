// util.hip - copy kernels: a plain streaming one (for calibrating byte
// counters: it reads and writes exactly `bytes` bytes once each) and the
// upload from pinned host memory.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "s2tc_internal.h"

namespace s2tc {

__global__ void k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16)
{
	for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x)
		dst[i] = src[i];
}

// Upload from mapped pinned memory, bound by the bus: 16 workgroups keep 256
// KiB of reads in flight and leave the other CUs to the encoders that run
// beside it.  Measured (MI355X): 8 MiB in 151 us, as the runtime's DMA engines
// (153 us), but a kernel of another stream that depends on it starts within 10
// us, and it on that one, where a DMA waits for 50 us and more.  64 workgroups
// are no faster alone, and 4096 x 4096 calls 15% slower for the encoder's wait.
#define PULL_WGS 16
__global__ __launch_bounds__(256) void k_pull(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n16)
{
	const size_t st = PULL_WGS * 256;
	size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
	for (; i + 3 * st < n16; i += 4 * st) {
		const uint4 a = src[i], b = src[i + st], c = src[i + 2 * st], d = src[i + 3 * st];
		dst[i] = a;
		dst[i + st] = b;
		dst[i + 2 * st] = c;
		dst[i + 3 * st] = d;
	}
	for (; i < n16; i += st) dst[i] = src[i];
}

int launch_pull(void *dst, const void *src, size_t n, hipStream_t st)
{
	k_pull<<<PULL_WGS, 256, 0, st>>>((const uint4 *)src, (uint4 *)dst, (n + 15) / 16);
	return hip_check(hipGetLastError(), "upload kernel");
}

}  // namespace s2tc

extern "C" int s2tc_amd_memcpy_d2d_kernel(void *dst, const void *src, size_t bytes, void *stream)
{
	using namespace s2tc;
	if (!dst || !src || (bytes & 15) || (((uintptr_t)dst | (uintptr_t)src) & 15))
		return set_error(S2TC_E_ARG, "copy kernel needs 16-byte aligned pointers and sizes");
	const size_t n16 = bytes / 16;
	const unsigned grid = (unsigned)((n16 + 255) / 256 < 65536 ? (n16 + 255) / 256 : 65536);
	k_copy16<<<grid ? grid : 1, 256, 0, (hipStream_t)stream>>>((const uint4 *)src, (uint4 *)dst, n16);
	return hip_check(hipGetLastError(), "copy kernel");
}
