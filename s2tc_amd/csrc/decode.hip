// decode.hip - S2TC block decoding and the total colour distance of an
// encoding, on the device.
//
// k_decode follows fetch_2d_texel_* (s2tc_libtxc_dxtn.cpp:35-140) for every
// texel of an image: index 0 / 1 take c0 / c1, indices 2 and 3 take the
// checkerboard of c0 and c1 (i ^ j odd -> c1), except DXT1 index 3 with
// c1 >= c0, which is black (alpha 0 for RGBA); 5:6:5 expands as (v << 3) |
// (v >> 2) and (v << 2) | (v >> 4); DXT3 alpha a | a << 4; DXT5 alpha in
// the 6-value mode (a1 >= a0: 6 -> 0, 7 -> 255, 6 falling through to 7's
// test otherwise) else the checkerboard.
//
// The colour-distance kernels live with the encoders (kernels_cd.hip),
// one per distance; s2tc_amd_colordist_error dispatches to them.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "s2tc_internal.h"

namespace s2tc {

__device__ __forceinline__ uint32_t expand565(uint32_t c)
{
	const uint32_t r = (c >> 11) & 31u, g = (c >> 5) & 63u, b = c & 31u;
	return ((r << 3) | (r >> 2)) | (((g << 2) | (g >> 4)) << 8) | (((b << 3) | (b >> 2)) << 16);
}

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x4_a1 __attribute__((ext_vector_type(4), aligned(1)));
typedef uint32_t u32x2_a1 __attribute__((ext_vector_type(2), aligned(1)));

// The four DXT5 alphas of a row, a byte each: idx holds its four 3-bit indices,
// even and odd the values of the eight indices for texels with i ^ j even and
// odd, four to a word.
__device__ __forceinline__ uint32_t row_alphas(uint32_t idx, const uint32_t (&even)[2], const uint32_t (&odd)[2], int y)
{
	const uint32_t sel = (idx & 7u) | ((idx & 0x38u) << 5) | ((idx & 0x1c0u) << 10) | ((idx & 0xe00u) << 15);
	const uint32_t e = __builtin_amdgcn_perm(even[1], even[0], sel), o = __builtin_amdgcn_perm(odd[1], odd[0], sel);
	const uint32_t m = (y & 1) ? 0x00ff00ffu : 0xff00ff00u;  // the odd texels of row y
	return (o & m) | (e & ~m);
}

// One lane per block: the block in one 8- or 16-byte load, its rows in four
// 16-byte stores (1 KiB of a texel row per wave and store).  All choices are
// bit masks and byte permutes, no branches.
//
// Bound: HBM, 4 B written per texel and 0.5 or 1 B read.  Measured (MI355X,
// 8192 x 8192 DXT5): 57 us = 5.9 TB/s; one lane per texel with byte loads took
// 201 us.
template <unsigned FMT>
__global__ __launch_bounds__(256) void k_decode(const uint8_t *__restrict__ blocks, int width, int height,
                                                uint32_t *__restrict__ rgba)
{
	const int bw = (width + 3) >> 2, bh = (height + 3) >> 2;
	const int bx = (int)(blockIdx.x * 64 + threadIdx.x), by = (int)(blockIdx.y * 4 + threadIdx.y);
	if (bx >= bw || by >= bh) return;
	constexpr bool DXT1 = FMT == 0x83F0u || FMT == 0x83F1u;
	const size_t b = (size_t)by * (size_t)bw + (size_t)bx;
	uint32_t ax = 0, ay = 0, cw, idx;
	if constexpr (DXT1) {
		const u32x2_a1 v = *(const u32x2_a1 *)(blocks + b * 8);
		cw = v[0];
		idx = v[1];
	} else {
		const u32x4_a1 v = *(const u32x4_a1 *)(blocks + b * 16);
		ax = v[0];
		ay = v[1];
		cw = v[2];
		idx = v[3];
	}
	const uint32_t c0 = cw & 0xffffu, c1 = cw >> 16;
	const uint32_t opaque = FMT == 0x83F0u || FMT == 0x83F1u ? 0xff000000u : 0u;
	const uint32_t e0 = expand565(c0) | opaque, diff = (expand565(c1) | opaque) ^ e0;
	// bit 2 k of these words is texel k = 4 y + x
	const uint32_t lo = idx & 0x55555555u, hi = (idx >> 1) & 0x55555555u;
	const uint32_t one = (lo & ~hi) | (hi & 0x11441144u);  // c1: index 1, or 2 and 3 with x ^ y odd
	const uint32_t black = DXT1 && c1 >= c0 ? lo & hi : 0u;
	const uint32_t none = FMT == 0x83F0u ? 0xff000000u : 0u;
	uint32_t even[2] = {0, 0}, odd[2] = {0, 0};
	if constexpr (FMT == 0x83F3u) {
		const uint32_t a0 = ax & 255u, a1 = (ax >> 8) & 255u;
		const bool six = a1 >= a0;
		const uint32_t r0 = a0 * 0x01010101u, r1 = a1 * 0x01010101u;
		even[0] = (r0 & 0xffff00ffu) | (a1 << 8);
		odd[0] = (r1 & 0xffffff00u) | a0;
		even[1] = six ? (r0 & 0xffffu) | 0xff000000u : r0;
		odd[1] = six ? (r1 & 0xffffu) | 0xff000000u : r1;
	}
	const int w = min(4, width - 4 * bx), h = min(4, height - 4 * by);
	uint32_t *o = rgba + (size_t)(4 * by) * (size_t)width + (size_t)(4 * bx);
#pragma unroll
	for (int y = 0; y < 4; ++y) {
		if (y >= h) break;
		uint32_t al = 0;  // the row's alphas, a byte each
		if constexpr (FMT == 0x83F2u) {
			const uint32_t n = ((y < 2 ? ax : ay) >> (16 * (y & 1))) & 0xffffu;
			const uint32_t s = (n & 15u) | ((n & 0xf0u) << 4) | ((n & 0xf00u) << 8) | ((n & 0xf000u) << 12);
			al = s | (s << 4);
		} else if constexpr (FMT == 0x83F3u) {
			// index bits 12 y .. 12 y + 11 of the 48 after the endpoints
			const uint32_t bits = y == 0   ? ax >> 16
			                      : y == 1 ? (ax >> 28) | (ay << 4)
			                      : y == 2 ? ay >> 8
			                               : ay >> 20;
			al = row_alphas(bits, even, odd, y);
		}
		u32x4_a4 t;
#pragma unroll
		for (int x = 0; x < 4; ++x) {
			const int k = 2 * (4 * y + x);
			uint32_t c = e0 ^ (diff & (0u - ((one >> k) & 1u)));
			if constexpr (DXT1) c = (black >> k) & 1u ? none : c;
			else c |= x == 3 ? al & 0xff000000u : (al << (24 - 8 * x)) & 0xff000000u;
			t[x] = c;
		}
		if (w == 4) {
			*(u32x4_a4 *)(o + (size_t)y * (size_t)width) = t;
		} else {
#pragma unroll
			for (int x = 0; x < 3; ++x)
				if (x < w) o[(size_t)y * (size_t)width + x] = t[x];
		}
	}
}

// ---- the sums of s2tc_amd_colordist_error ----

// A call's pinned words for the workgroups' sums, kept for later calls on the
// same device (allocating and clearing a device word took 25 us a call).  A
// call owns its buffer from acquire to release, so calls from several threads
// or on several streams do not meet.
static const unsigned kSumsMax = 512;
struct SumBuf {
	int dev;
	long long *sums, *dev_sums;  // [kSumsMax]
};

static std::mutex g_sum_mu;
static std::vector<SumBuf *> g_sums;
static const size_t kSumBufsKept = 16;

static int sum_acquire(SumBuf **out)
{
	int dev = 0;
	if (int r = hip_check(hipGetDevice(&dev), "hipGetDevice")) return r;
	{
		std::lock_guard<std::mutex> lk(g_sum_mu);
		for (size_t i = 0; i < g_sums.size(); ++i)
			if (g_sums[i]->dev == dev) {
				*out = g_sums[i];
				g_sums[i] = g_sums.back();
				g_sums.pop_back();
				return 0;
			}
	}
	SumBuf *b = new SumBuf{dev, nullptr, nullptr};
	int rc = hip_check(hipHostMalloc((void **)&b->sums, kSumsMax * sizeof(long long), hipHostMallocMapped),
	                   "hipHostMalloc");
	if (!rc) rc = hip_check(hipHostGetDevicePointer((void **)&b->dev_sums, b->sums, 0), "hipHostGetDevicePointer");
	if (rc) {
		if (b->sums) (void)hipHostFree(b->sums);
		delete b;
		return rc;
	}
	*out = b;
	return 0;
}

static void sum_release(SumBuf *b)
{
	{
		std::lock_guard<std::mutex> lk(g_sum_mu);
		if (g_sums.size() < kSumBufsKept) {
			g_sums.push_back(b);
			return;
		}
	}
	(void)hipHostFree(b->sums);
	delete b;
}

}  // namespace s2tc

using namespace s2tc;

extern "C" int s2tc_amd_decode_image(const void *d_blocks, unsigned int format, int width, int height, void *d_rgba,
                                     void *stream)
{
	if (!d_blocks || !d_rgba || width <= 0 || height <= 0)
		return set_error(S2TC_E_ARG, "decode: bad arguments");
	if (format < 0x83F0u || format > 0x83F3u) return set_error(S2TC_E_ARG, "decode: bad format 0x%x", format);
	if (int r = ensure_device()) return r;
	const int by = (height + 3) / 4;
	if (by > 65535) return set_error(S2TC_E_RANGE, "decode: image too tall");
	const int bw = (width + 3) / 4;
	const dim3 grid((unsigned)((bw + 63) / 64), (unsigned)((by + 3) / 4)), block(64, 4);
	hipStream_t st = (hipStream_t)stream;
	const uint8_t *in = (const uint8_t *)d_blocks;
	uint32_t *out = (uint32_t *)d_rgba;
	if (format == 0x83F0u) k_decode<0x83F0u><<<grid, block, 0, st>>>(in, width, height, out);
	else if (format == 0x83F1u) k_decode<0x83F1u><<<grid, block, 0, st>>>(in, width, height, out);
	else if (format == 0x83F2u) k_decode<0x83F2u><<<grid, block, 0, st>>>(in, width, height, out);
	else k_decode<0x83F3u><<<grid, block, 0, st>>>(in, width, height, out);
	return hip_check(hipGetLastError(), "launch k_decode");
}

extern "C" int s2tc_amd_colordist_error(const void *d_src, int src_kind, int width, int height, const void *d_blocks,
                                        int dxt, int cd, long long *total, void *stream)
{
	if (!d_src || !d_blocks || !total || width <= 0 || height <= 0)
		return set_error(S2TC_E_ARG, "colordist_error: bad arguments");
	if (src_kind != S2TC_SRC_QUANTIZED && src_kind != S2TC_SRC_RGBA8)
		return set_error(S2TC_E_ARG, "colordist_error: bad source kind %d", src_kind);
	int refine = REFINE_ALWAYS;
	normalize_modes(dxt, cd, refine);
	if (int r = ensure_device()) return r;
	const KernelTable &kt = kernel_table(cd);
	const void *k = kt.error[dxt][src_kind == S2TC_SRC_RGBA8 ? 1 : 0];
	if (!k) return set_error(S2TC_E_ARG, "colordist_error: no kernel for distance %d", cd);
	const int bw = (width + 3) / 4, bh = (height + 3) / 4;
	if (bh > 4 * 65535) return set_error(S2TC_E_RANGE, "colordist_error: image too tall");
	hipStream_t st = (hipStream_t)stream;
	SumBuf *b = nullptr;
	if (int r = sum_acquire(&b)) return r;
	const long long tiles = (long long)((bw + 63) / 64) * ((bh + 3) / 4);
	// two workgroups per CU hide each other's loads
	const unsigned grid = (unsigned)std::min<long long>(tiles, kSumsMax);
	void *args[] = {(void *)&d_src, (void *)&width, (void *)&height, (void *)&d_blocks, (void *)&b->dev_sums};
	int rc = hip_check(hipLaunchKernel(k, dim3(grid), dim3(64, 4), args, 0, st), "launch colour-distance kernel");
	// also after a failed launch: nothing may still write to the buffer
	const int rs = hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
	if (!rc) rc = rs;
	if (!rc) {
		long long sum = 0;
		for (unsigned i = 0; i < grid; ++i) sum += b->sums[i];
		*total = sum;
	}
	sum_release(b);
	return rc;
}
