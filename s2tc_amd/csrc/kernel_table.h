// kernel_table.h - per-distance-mode table of encoder kernels (host side).
#pragma once

#include <cstddef>
#include <cstdint>

// One image (a texture's mip level) of a batch, as the persistent kernels see it.
struct JobDesc {
	const uint32_t *src;  // width*height texels, 4 bytes each
	uint8_t *dst;         // blocks in raster order
	int width, height;
	int dxt, nrandom, refine, raw;  // raw: RGBA8 quantized on load with DITHER_NONE
	unsigned long long seed;
	long long block0;     // first block of this job in its class's packed block index space
	uint32_t bw_magic;    // min(2^32 / bw, 2^32 - 1) for bw = block columns: see div_blocks
	uint32_t pad;
};

// The multiplier of div_blocks for bw block columns (bw >= 1).
inline uint32_t bw_magic(int bw)
{
	const unsigned long long m = (1ull << 32) / (unsigned long long)bw;
	return m > 0xffffffffull ? 0xffffffffu : (uint32_t)m;
}

// First and last job index a batch tile touches.
struct TileJobs {
	int lo, hi;
};

struct KernelTable {
	const void *fast[3][2][3][2];  // [dxt][raw][refine][edge]: k_fast_interior (full blocks; edge: and partial ones), null for NORMALMAP
	const void *normal[2][2];     // [many][raw]: k_normal<CD, raw, RB> (many: normal_many)
	const void *normal_wide[2];   // [raw]: k_normal_wide<CD, raw> (group memory in global scratch)
	int normal_smem_cand;         // LDS bytes per candidate slot of a 4-block workgroup (candidate words)
	int normal_smem_fixed;        // plus these bytes (features of the 16 texel candidates of 4 blocks)
	const void *fast_batch[3][3]; // [dxt][refine]: persistent quick-mode kernel over a job list
	const void *normal_batch[2];  // [many]: persistent MODE_NORMAL kernel over a job list (many: class_many)
	const void *normal_batch_wide;  // the same with group memory in global scratch
	const void *all16[3][2];      // [dxt][raw]: MODE_NORMAL without random colours, one lane per block
	const void *all16_batch[3][3];  // [dxt][refine]: its persistent batch form
	const void *all16_batch_alone[3][3];  // the form for a batch of this one class
	const void *error[3][2];      // [dxt][raw]: k_colordist_error (total colour distance of an encoding)
	const void *init;             // per-device table set-up kernel (256 x 256 threads, one int argument), or null
	const void *set_scan_cap;     // k_set_scan_cap (one workgroup of 64 threads, one uint32_t argument)
};

// Row blocks (16 rows each) of a block's distance matrix that the
// random-candidate kernels keep in registers instead of group memory.  The
// kernels with two run four waves to a SIMD.  From five row blocks to eight
// (49 to 112 random colours) group memory holds fewer workgroups than that, 11
// to 6 to a CU, which the SIMDs share unevenly; with three row blocks in 168
// registers twelve to 8 fit.  Measured (MI355X, 1024 x 1024, two -> three):
// NORMALMAP 64 random colours 134.9 -> 117.4 us, 112 267 -> 235 us; SRGB 337 ->
// 278 us and 1075 -> 975 us.  Outside that range, and where a launch has no
// more workgroups than eight to a CU, the third row block only costs moves:
// 48 random colours up to 8% slower, 128 SRGB 2%, 256 x 256 SRGB 8%.
#define S2TC_RB_FEW 2
#define S2TC_RB_MANY 3
inline bool normal_many(int pbw, long long workgroups, int cus)
{
	return pbw >= 5 && pbw <= 8 && workgroups > 8LL * cus;
}

// A class of a batch takes textures of all counts: three row blocks where three
// quarters of its pair work (blocks times row blocks squared) lie in that range.
// Measured (40 textures of 256 x 256 with few random colours and some with 64,
// the class alone, two and three): SRGB 8 and one 64 401 and 456 us, 16 and ten
// 64 697 and 760 us; NORMALMAP alike with both.  Only 64 random colours, 4
// workgroups a CU: RGB 5% slower with three, SRGB 2%, the others within 1%; but
// with as many as fit a CU, as in a tuned batch, faster: the YUV class of the
// serving pool 2.88 and 2.12 ms, the pool as one batch 4.56 and 3.97 ms.
inline bool class_many(double many_work, double work, int pbw_max, long long workgroups, int cus)
{
	return normal_many(pbw_max, workgroups, cus) && 4 * many_work >= 3 * work;
}

#if defined(__HIP__) || defined(__HIPCC__)
#define S2TC_HD __host__ __device__
#else
#define S2TC_HD
#endif

// Ints of row memory per block with pbw row blocks, rb of them in registers:
// the other rows.  With three in registers and five in all, 560 instead of
// 512, so that the tables of the scan over distinct colours hold a box of 160
// cells (two ints a cell, three a candidate): 80 candidates fall on 63 of
// them, a row block less, and twelve workgroups still fit a CU.  Measured: a 4096 x
// 4096 normal map with 64 random colours 499 -> 491 us; 1024 x 1024 with 49 to 64
// under five distances and three contents within 1.5% either way, 1.000 on average.
S2TC_HD inline int normal_row_ints(int pbw, int rb)
{
	const int rows = 256 * (pbw > rb ? pbw - rb : 0);
	return rb == S2TC_RB_MANY && rows < 560 ? 560 : rows;
}

// Ints of a block's row memory (`ints` in all) that the tables of the scan over
// distinct colours and its list may take: no more than the rows of the block's
// own pbw row blocks with two in registers, also where the launch was sized for
// larger blocks of its class.  Blocks with few candidates have little to gain:
// 40 textures with 16 random colours and 10 with 64 (256 x 256, NORMALMAP, boxes
// of 30 to 250 cells) took 651 us with tables in all that the class has, 576 us
// so; RGB 654 and 592 us.
S2TC_HD inline int normal_table_ints(int pbw, int ints)
{
	const int own = 256 * (pbw > S2TC_RB_FEW ? pbw - S2TC_RB_FEW : 0);
	return own < ints ? own : ints;
}

// Group memory of a four-block workgroup of the random-candidate kernels
// with pbw row blocks: 16 pbw candidate slots, the row memory and the texel
// features.
inline size_t normal_group_smem(const KernelTable &kt, int pbw, bool many)
{
	const int rb = many ? S2TC_RB_MANY : S2TC_RB_FEW;
	return (size_t)kt.normal_smem_cand * 16 * (size_t)pbw +
	       (size_t)4 * sizeof(int) * (size_t)normal_row_ints(pbw, rb) + (size_t)kt.normal_smem_fixed;
}

extern "C" {
void s2tc_kernels_cd0(KernelTable *);
void s2tc_kernels_cd1(KernelTable *);
void s2tc_kernels_cd2(KernelTable *);
void s2tc_kernels_cd3(KernelTable *);
void s2tc_kernels_cd4(KernelTable *);
void s2tc_kernels_cd5(KernelTable *);
void s2tc_kernels_cd6(KernelTable *);
void s2tc_kernels_cd7(KernelTable *);
}
