// s2tc_internal.h - shared declarations of the host-side library code.
#pragma once

#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__ 1
#endif
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <cstdint>

#include "kernel_table.h"
#include "s2tc_amd.h"

namespace s2tc {

enum { DXT1 = 0, DXT3 = 1, DXT5 = 2 };
enum { REFINE_NEVER = 0, REFINE_ALWAYS = 1, REFINE_LOOP = 2 };
enum { CD_RGB = 0, CD_YUV = 1, CD_SRGB = 2, CD_SRGB_MIXED = 3, CD_AVG = 4, CD_WAVG = 5, CD_W0AVG = 6,
       CD_NORMALMAP = 7 };
enum { DITHER_NONE = 0, DITHER_SIMPLE = 1, DITHER_FLOYDSTEINBERG = 2 };

struct EncodeArgs {
	const void *src;
	void *dst;
	int src_kind;
	int width, height;
	int dxt, cd, nrandom, refine;
	uint64_t seed;
	uint32_t block_index_base;  // generator block index of the image's first block
};

int set_error(int code, const char *fmt, ...);
int hip_check(hipError_t e, const char *what);
int ensure_device();
const KernelTable &kernel_table(int cd);
void normalize_modes(int &dxt, int &cd, int &refine);
bool is_fast(int cd, int nrandom);
int normal_pbw(int nrandom);
// Encodes one image on `stream`.  Random-candidate encodes above
// S2TC_LDS_NRANDOM need device scratch: from `ext_scratch` (ext_bytes long;
// the grid shrinks to what fits) when given, else allocated stream-ordered
// around the launch.
int launch_encode(const EncodeArgs &a, hipStream_t stream, void *ext_scratch = nullptr, size_t ext_bytes = 0);

// Upload from pinned host memory by its device address (util.hip): n bytes
// rounded up to 16, which both buffers hold, at 16-byte aligned addresses.
int launch_pull(void *dst, const void *src, size_t n, hipStream_t st);

// rgb565_image on the device (dither.hip); d_scratch holds
// rgb565_scratch_bytes(w, h, dither).
// d_carry_in / d_carry_out (4 bytes each, apart; SIMPLE only): the image is a
// band of rows of a larger one, which starts from the error states in
// d_carry_in (null: from the reference's initial ones) and leaves its end
// states in d_carry_out for the next band.
// host_src: d_src is pinned host memory, worth reading once only; d_out is then
// 16-byte aligned.
// fs: a run of the Floyd-Steinberg dither.  Its waves wait for each other:
// gave_up, a word in mapped pinned memory that the caller clears before, is 1
// after the launch if one of them ended without what it waited for, and the
// output is then wrong; polls bounds each wait (FS_POLLS looks at memory take
// seconds).  slab bounds the scratch for channel planes, of which one band of 64
// rows is the least (512 bytes a column); less than the image needs costs the
// time to drain and fill the wavefront between slabs.
static const unsigned FS_POLLS = 1u << 22;
static const size_t FS_SLAB = (size_t)512 << 20;
struct FsRun {
	uint32_t *gave_up = nullptr;
	unsigned polls = FS_POLLS;
	size_t slab = FS_SLAB;
};
size_t rgb565_scratch_bytes(int w, int h, int dither, size_t fs_slab = FS_SLAB);
int launch_rgb565(const void *d_src, int srccomps, int w, int h, int alphabits, int dither, void *d_out,
                  void *d_scratch, hipStream_t st, const void *d_carry_in = nullptr, void *d_carry_out = nullptr,
                  bool host_src = false, const FsRun &fs = FsRun());

// The Floyd-Steinberg dither (dither_fs.hip), arguments normalised.
size_t rgb565_fs_scratch_bytes(int w, int h, size_t slab);
int launch_rgb565_fs(const uint8_t *src, int srccomps, int w, int h, int alphabits, uint8_t *out, void *d_scratch,
                     hipStream_t st, const FsRun &run);

inline int block_bytes(int dxt) { return dxt == DXT1 ? 8 : 16; }

}  // namespace s2tc

