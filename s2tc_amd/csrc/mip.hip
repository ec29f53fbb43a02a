// mip.hip - the CLI's mip chain on the device.
//
// Image_MipReduce32 (s2tc_compress.c:427-493) halves an RGBA8 image with a
// truncating box filter: both sides > 1 -> (a + b + c + d) >> 2 over 2x2,
// only the width > 1 -> (a + b) >> 1 over horizontal pairs, only the height
// > 1 -> (a + b) >> 1 over vertical pairs; odd last rows / columns are
// dropped (the new size is the old size >> 1).  The chain of
// s2tc_compress.c:722-733 repeats it down to 1x1.  The four channels are
// summed in 16-bit lanes of two words.  A single halving and the batch's
// levels take one thread per output texel; a chain takes six levels per
// launch (k_mip_levels).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

#include "s2tc_internal.h"

namespace s2tc {

// per-channel sum of RGBA8 words in two words of 16-bit lanes (r|b, g|a)
struct Sum4 {
	uint32_t rb, ga;
	__device__ __forceinline__ void add(uint32_t p)
	{
		rb += p & 0x00ff00ffu;
		ga += (p >> 8) & 0x00ff00ffu;
	}
	__device__ __forceinline__ uint32_t shifted(int s) const
	{
		return ((rb >> s) & 0x00ff00ffu) | (((ga >> s) & 0x00ff00ffu) << 8);
	}
};

__device__ __forceinline__ void mip_texel(const uint32_t *__restrict__ in, int width, int height,
                                          uint32_t *__restrict__ out, int x, int y, int ow);

__global__ __launch_bounds__(256) void k_mip_reduce(const uint32_t *__restrict__ in, int width, int height,
                                                    uint32_t *__restrict__ out)
{
	const int ow = width > 1 ? width >> 1 : 1, oh = height > 1 ? height >> 1 : 1;
	const int x = (int)(blockIdx.x * 64 + threadIdx.x), y = (int)(blockIdx.y * 4 + threadIdx.y);
	if (x >= ow || y >= oh) return;
	mip_texel(in, width, height, out, x, y, ow);
}

// One level of many chains in one launch: a task is one texture's halving
// at this level; tasks own consecutive runs of 256-texel tiles (tile0 is the
// first), and a workgroup finds its task by a binary search over tile0.
struct MipTask {
	const uint32_t *in;
	uint32_t *out;
	int w, h;          // input size
	uint32_t tile0;
	uint32_t pad;
};

__device__ __forceinline__ void mip_texel(const uint32_t *__restrict__ in, int width, int height,
                                          uint32_t *__restrict__ out, int x, int y, int ow)
{
	Sum4 s{0u, 0u};
	int shift;
	if (width > 1 && height > 1) {
		const uint32_t *r0 = in + (size_t)(2 * y) * (size_t)width + 2 * x, *r1 = r0 + width;
		s.add(r0[0]);
		s.add(r0[1]);
		s.add(r1[0]);
		s.add(r1[1]);
		shift = 2;
	} else if (width > 1) {
		const uint32_t *r0 = in + (size_t)y * (size_t)width + 2 * x;
		s.add(r0[0]);
		s.add(r0[1]);
		shift = 1;
	} else {
		const uint32_t *r0 = in + (size_t)(2 * y) * (size_t)width + x;
		s.add(r0[0]);
		s.add(r0[width]);
		shift = 1;
	}
	out[(size_t)y * (size_t)ow + x] = s.shifted(shift);
}

// Six levels of one chain: a workgroup reads a 64 x 64 tile of level 0 and
// writes its part of levels 1 to 6 (and level 0 itself if base0 is set: the
// image is copied into the chain).  Tiles start at multiples of 64, so what a
// tile's texels are made of lies in the tile at every level, odd sizes (whose
// last row or column is dropped) and sides of 1 included.  Each lane reduces
// its 4 x 4 texels twice in registers, the rest goes through LDS.
//
// Bound: HBM, each texel of level 0 read once and every level written once (a
// launch per level reads each level again, and a copy level 0 twice).
// Measured (MI355X, 4096 x 4096 into another buffer): 25 us for the first six
// levels = 6 TB/s and 4 us for the rest, the call 38 us; a copy and twelve
// launches took 64 us.
struct MipLevels {
	const uint32_t *in;
	uint32_t *out[7];  // levels 0 (or null) to 6; null past the last one
	int w, h;
};

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));

// (a b / c d) to one texel; wide, tall: the level has pairs of columns, rows.
__device__ __forceinline__ uint32_t mip_quad(uint32_t a, uint32_t b, uint32_t c, uint32_t d, bool wide, bool tall)
{
	Sum4 s{0u, 0u};
	s.add(a);
	if (wide) s.add(b);
	if (tall) s.add(c);
	if (wide && tall) s.add(d);
	return s.shifted((wide ? 1 : 0) + (tall ? 1 : 0));
}

__global__ __launch_bounds__(256) void k_mip_levels(MipLevels m)
{
	__shared__ uint32_t lds[16 * 17];
	const int tx = (int)(threadIdx.x & 15), ty = (int)(threadIdx.x >> 4);
	int w = m.w, h = m.h;
	const int x0 = (int)blockIdx.x * 64 + 4 * tx, y0 = (int)blockIdx.y * 64 + 4 * ty;
	uint32_t t[4][4];
	const int nx = min(4, w - x0), ny = min(4, h - y0);  // may be negative
#pragma unroll
	for (int y = 0; y < 4; ++y) {
#pragma unroll
		for (int x = 0; x < 4; ++x) t[y][x] = 0;
		if (y >= ny || nx <= 0) continue;
		const size_t at = (size_t)(y0 + y) * (size_t)w + (size_t)x0;
		if (nx == 4) {
			const u32x4_a4 v = *(const u32x4_a4 *)(m.in + at);
#pragma unroll
			for (int x = 0; x < 4; ++x) t[y][x] = v[x];
			if (m.out[0]) *(u32x4_a4 *)(m.out[0] + at) = v;
		} else {
#pragma unroll
			for (int x = 0; x < 3; ++x)
				if (x < nx) {
					t[y][x] = m.in[at + x];
					if (m.out[0]) m.out[0][at + x] = t[y][x];
				}
		}
	}
	if (!m.out[1]) return;
	// level 1: 2 x 2 of the lane
	bool wide = w > 1, tall = h > 1;
	w = wide ? w >> 1 : 1;
	h = tall ? h >> 1 : 1;
	uint32_t u[2][2];
	const int x1 = x0 >> 1, y1 = y0 >> 1;
#pragma unroll
	for (int y = 0; y < 2; ++y) {
#pragma unroll
		for (int x = 0; x < 2; ++x)
			u[y][x] = mip_quad(t[2 * y][2 * x], t[2 * y][2 * x + 1], t[2 * y + 1][2 * x], t[2 * y + 1][2 * x + 1], wide, tall);
		if (y1 + y >= h) continue;
		uint32_t *o = m.out[1] + (size_t)(y1 + y) * (size_t)w + (size_t)x1;
		if (x1 + 1 < w) *(u32x2_a4 *)o = u32x2_a4{u[y][0], u[y][1]};
		else if (x1 < w) o[0] = u[y][0];
	}
	if (!m.out[2]) return;
	// level 2: one texel of the lane
	wide = w > 1, tall = h > 1;
	w = wide ? w >> 1 : 1;
	h = tall ? h >> 1 : 1;
	uint32_t v = mip_quad(u[0][0], u[0][1], u[1][0], u[1][1], wide, tall);
	if (x0 >> 2 < w && y0 >> 2 < h) m.out[2][(size_t)(y0 >> 2) * (size_t)w + (size_t)(x0 >> 2)] = v;
	// levels 3 to 6: the tile's 8 x 8, 4 x 4, 2 x 2 and 1 texels, one lane each
	lds[ty * 17 + tx] = v;
#pragma unroll
	for (int l = 3; l <= 6; ++l) {
		if (!m.out[l]) return;
		const int n = 64 >> l;  // texels of the tile's side at this level
		wide = w > 1, tall = h > 1;
		w = wide ? w >> 1 : 1;
		h = tall ? h >> 1 : 1;
		__syncthreads();
		const bool mine = tx < n && ty < n;
		if (mine) {
			const uint32_t *p = lds + 2 * ty * 17 + 2 * tx;
			v = mip_quad(p[0], p[1], p[17], p[18], wide, tall);
			const int x = (int)blockIdx.x * n + tx, y = (int)blockIdx.y * n + ty;
			if (x < w && y < h) m.out[l][(size_t)y * (size_t)w + (size_t)x] = v;
		}
		__syncthreads();
		if (mine) lds[ty * 17 + tx] = v;
	}
}

__global__ __launch_bounds__(256) void k_mip_reduce_batch(const MipTask *__restrict__ tasks, int ntasks)
{
	const uint32_t tile = blockIdx.x;
	int lo = 0, hi = ntasks - 1;
	while (lo < hi) {
		const int mid = (lo + hi + 1) >> 1;
		if (tasks[mid].tile0 <= tile) lo = mid;
		else hi = mid - 1;
	}
	const MipTask t = tasks[lo];
	const int ow = t.w > 1 ? t.w >> 1 : 1, oh = t.h > 1 ? t.h >> 1 : 1;
	const uint32_t i = (tile - t.tile0) * 256u + threadIdx.x;
	if (i >= (uint32_t)ow * (uint32_t)oh) return;
	const int y = (int)(i / (uint32_t)ow), x = (int)(i - (uint32_t)y * (uint32_t)ow);
	mip_texel(t.in, t.w, t.h, t.out, x, y, ow);
}

}  // namespace s2tc

using namespace s2tc;

static size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

extern "C" int s2tc_amd_mip_layout(int width, int height, int *nlevels, size_t *offsets, int *widths, int *heights,
                                   int max_levels, size_t *total_bytes)
{
	if (width <= 0 || height <= 0 || !nlevels) return set_error(S2TC_E_ARG, "mip_layout: bad arguments");
	int w = width, h = height, n = 0;
	size_t off = 0;
	for (;;) {
		if (n < max_levels) {
			if (offsets) offsets[n] = off;
			if (widths) widths[n] = w;
			if (heights) heights[n] = h;
		}
		off += align256((size_t)w * h * 4);
		++n;
		if (w == 1 && h == 1) break;
		w = w > 1 ? w >> 1 : 1;
		h = h > 1 ? h >> 1 : 1;
	}
	*nlevels = n;
	if (total_bytes) *total_bytes = off;
	return 0;
}

extern "C" int s2tc_amd_mip_reduce(const void *d_in, int width, int height, void *d_out, void *stream)
{
	if (!d_in || !d_out || width <= 0 || height <= 0) return set_error(S2TC_E_ARG, "mip_reduce: bad arguments");
	if (width == 1 && height == 1) return set_error(S2TC_E_ARG, "mip_reduce: the image is already 1x1");
	if (int r = ensure_device()) return r;
	const int ow = width > 1 ? width >> 1 : 1, oh = height > 1 ? height >> 1 : 1;
	if ((oh + 3) / 4 > 65535) return set_error(S2TC_E_RANGE, "mip_reduce: image too tall");
	dim3 grid((unsigned)((ow + 63) / 64), (unsigned)((oh + 3) / 4)), block(64, 4);
	k_mip_reduce<<<grid, block, 0, (hipStream_t)stream>>>((const uint32_t *)d_in, width, height, (uint32_t *)d_out);
	return hip_check(hipGetLastError(), "launch k_mip_reduce");
}

extern "C" int s2tc_amd_mip_chain(const void *d_src, int width, int height, void *d_levels, size_t capacity,
                                  void *stream)
{
	int n = 0;
	size_t total = 0;
	if (int r = s2tc_amd_mip_layout(width, height, &n, nullptr, nullptr, nullptr, 0, &total)) return r;
	if (!d_src || !d_levels) return set_error(S2TC_E_ARG, "mip_chain: null buffer");
	if (capacity < total) return set_error(S2TC_E_ARG, "mip_chain: %zu bytes needed, %zu given", total, capacity);
	if (int r = ensure_device()) return r;
	if ((height >> 1) + 3 >= 4 * 65536) return set_error(S2TC_E_RANGE, "mip_reduce: image too tall");
	hipStream_t st = (hipStream_t)stream;
	uint8_t *base = (uint8_t *)d_levels;
	if (n == 1) {
		if (d_src == d_levels) return n;
		if (int r = hip_check(hipMemcpyAsync(base, d_src, 4, hipMemcpyDeviceToDevice, st), "D2D")) return r;
		return n;
	}
	const uint32_t *in = (const uint32_t *)d_src;
	const uintptr_t s0 = (uintptr_t)d_src, d0 = (uintptr_t)d_levels;
	const size_t bytes = (size_t)width * height * 4;
	if (s0 != d0 && s0 < d0 + total && d0 < s0 + bytes) {
		// a source where levels go: copied before any is written
		if (int r = hip_check(hipMemcpyAsync(base, d_src, bytes, hipMemcpyDeviceToDevice, st), "D2D")) return r;
		in = (const uint32_t *)base;
	}
	int w = width, h = height;
	size_t off = 0;
	for (int l0 = 0; l0 < n - 1; l0 += 6) {
		// levels l0 + 1 .. l0 + 6 from level l0; the first launch also places level 0
		MipLevels m{};
		m.in = in;
		m.w = w;
		m.h = h;
		if (l0 == 0 && (const uint8_t *)in != base) m.out[0] = (uint32_t *)base;
		const dim3 grid((unsigned)((w + 63) / 64), (unsigned)((h + 63) / 64));
		for (int l = 1; l <= 6 && l0 + l < n; ++l) {
			off += align256((size_t)w * h * 4);
			m.out[l] = (uint32_t *)(base + off);
			w = w > 1 ? w >> 1 : 1;
			h = h > 1 ? h >> 1 : 1;
		}
		in = (const uint32_t *)(base + off);
		k_mip_levels<<<grid, 256, 0, st>>>(m);
		if (int r = hip_check(hipGetLastError(), "launch k_mip_levels")) return r;
	}
	return n;
}

extern "C" int s2tc_amd_mip_chain_batch(const s2tc_amd_mip_job *jobs, int njobs, void *stream)
{
	if (njobs < 0 || (njobs && !jobs)) return set_error(S2TC_E_ARG, "mip_chain_batch: bad arguments");
	// per texture: level offsets and sizes; then the tasks of every level
	std::vector<std::vector<MipTask>> levels;
	for (int j = 0; j < njobs; ++j) {
		const s2tc_amd_mip_job &jb = jobs[j];
		if (!jb.levels || jb.width <= 0 || jb.height <= 0)
			return set_error(S2TC_E_ARG, "mip_chain_batch: job %d: bad image", j);
		int w = jb.width, h = jb.height, l = 0;
		size_t off = 0;
		while (!(w == 1 && h == 1)) {
			const size_t next = off + align256((size_t)w * h * 4);
			if ((size_t)l >= levels.size()) levels.emplace_back();
			MipTask t;
			t.in = (const uint32_t *)((const uint8_t *)jb.levels + off);
			t.out = (uint32_t *)((uint8_t *)jb.levels + next);
			t.w = w;
			t.h = h;
			t.tile0 = 0;
			t.pad = 0;
			levels[l].push_back(t);
			off = next;
			w = w > 1 ? w >> 1 : 1;
			h = h > 1 ? h >> 1 : 1;
			++l;
		}
	}
	if (levels.empty()) return 0;
	std::vector<size_t> first(levels.size());
	std::vector<uint32_t> ntiles(levels.size());
	std::vector<MipTask> all;
	for (size_t l = 0; l < levels.size(); ++l) {
		uint64_t tiles = 0;
		for (MipTask &t : levels[l]) {
			t.tile0 = (uint32_t)tiles;
			const uint64_t ow = t.w > 1 ? t.w >> 1 : 1, oh = t.h > 1 ? t.h >> 1 : 1;
			tiles += (ow * oh + 255) / 256;
		}
		if (tiles > 0x7fffffffull) return set_error(S2TC_E_RANGE, "mip_chain_batch: level %zu too large", l);
		first[l] = all.size();
		ntiles[l] = (uint32_t)tiles;
		all.insert(all.end(), levels[l].begin(), levels[l].end());
	}
	if (int r = ensure_device()) return r;
	hipStream_t st = (hipStream_t)stream;
	MipTask *d = nullptr;
	int rc = hip_check(hipMalloc((void **)&d, all.size() * sizeof(MipTask)), "hipMalloc mip tasks");
	if (!rc)
		rc = hip_check(hipMemcpyAsync(d, all.data(), all.size() * sizeof(MipTask), hipMemcpyHostToDevice, st),
		               "H2D mip tasks");
	for (size_t l = 0; !rc && l < levels.size(); ++l) {
		k_mip_reduce_batch<<<ntiles[l], 256, 0, st>>>(d + first[l], (int)levels[l].size());
		rc = hip_check(hipGetLastError(), "launch k_mip_reduce_batch");
	}
	// the task list is read by the kernels: keep it until they are done
	const int rs = hip_check(hipStreamSynchronize(st), "mip_chain_batch synchronize");
	if (d) (void)hipFree(d);
	return rc ? rc : rs;
}
