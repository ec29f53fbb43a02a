// dither_fs.hip - the Floyd-Steinberg dither of rgb565_image on the GPU
// (s2tc_algorithm.cpp:1196-1267, 1350-1412).
//
// Every texel (x, y) adds its error sum to a 12-bit source value, quantizes
// it and splits the new error into e7 (right), e3, e5, e1 (below left, below,
// below right): acc(x, y) = e7(x - 1, y) + A_y[x + 1], where A_{y+1}[x] =
// e1(x - 2, y) + e5(x - 1, y) + e3(x, y) is final once row y has done texel
// x.  So row y may run two texels behind row y - 1, and the whole pass is a
// wavefront of w + 2 h steps with a short serial chain in each.
//
// Bound: that chain, at one wave per SIMD 4 cycles an instruction whether or
// not it depends on the one before, so the count of instructions per step is
// what matters.  A row is one lane: a wave owns a band of 64 rows, lane r at
// step t works on texel x = t - 2 r, and A_{y+1} moves to the next lane with
// one wave shift per step (no barrier).  Lane 63 hands its sums to lane 0 of
// the next band's wave, 8 at a time: through LDS inside a workgroup of four
// bands (one wave on each SIMD of a CU), through global memory to the next
// workgroup, on another CU.  The words themselves are the flags (they start
// as NO_CARRY, which no sum is).  Workgroups take their bands from a counter,
// so a wave only waits for waves that already run.  The arithmetic is exact
// in fp32 (all values are integers of a few thousand), where a truncating
// division is one fma and one trunc.
//
// The source values travel as planes of halves, one per channel, in the order
// the waves read them (slot [band][t / 8][row] of 8 steps: a wave's load is 1
// KiB); a step's quantized values go back into the first half of their slot,
// and a last kernel interleaves the channels.
//
// Measured (MI355X, RGBA, alpha copied): 1024 x 1024 0.22 ms, 4096 x 4096 0.80
// ms; k_fs_rows takes 68 ns a step at 1024 x 1024 (209 us; the alpha pass with one
// channel 56 ns, 174 us), where the waves of each band still start up for much of
// the time, and 47 ns at 4096 x 4096.  One workgroup per channel with a barrier per
// step took 2.3 ms and 37 ms; carries through global memory alone 0.21 and 0.89 ms.
//
// Memory: the planes take 8 bytes a texel and a band of 64 rows 512 a column and
// 80 KiB, in slabs of up to FS_SLAB; rows of a few texels are padded to 160 steps.
//
// The reference reuses one error buffer for the colour and the alpha pass and
// does not clear the part the alpha pass reads for its first row: that row
// starts from the red-channel errors the colour pass left there (the sums
// the last row read when h - 1 is even, else that row's downward errors).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>

#include "s2tc_internal.h"

namespace s2tc {

#define FS_ROWS 64              // rows of a band: the lanes of a wave
#define FS_STEP 8               // steps of a slot
#define FS_LAG (2 * (FS_ROWS - 1))  // lane 63's lag behind lane 0 in steps
#define FS_AHEAD 4              // slots loaded ahead of the one in work
#define FS_ZERO_GROUPS (2 * FS_AHEAD)  // zeros read by the lanes that get no carries
#define FS_WAVES 4              // bands of a workgroup: one wave on each SIMD of a CU
#define FS_LDS_MAX (156 << 10)  // LDS of a workgroup: rows of up to FS_LDS_WIDTH texels
#define NO_CARRY 0xffffffffu    // a carry word that is not there yet (a NaN)

// A wave's last slot lies at most FS_LAG steps and a round of FS_AHEAD after
// its last carry group, and groups are loaded ahead: what is allocated past
// the carries so that those loads, which are not used, stay inside.
#define FS_PAD_WORDS (FS_STEP * ((FS_LAG + 2) / FS_STEP + 2 * FS_AHEAD + 2))

// A wave only waits for waves with smaller tickets, which run.  Should a wait
// all the same last longer than FsRun::polls looks at memory or FS_LDS_POLLS
// times as many at LDS (a microsecond and a tenth of one each), the wave takes
// zeros for the missing sums, sets FsRun::gave_up, which makes the call an
// error, and waits no more, so that every wave still ends.
#define FS_LDS_POLLS 8

struct FsDims {
	int w;         // texels per row
	int y0, rows;  // this slab of the image
	int nb;        // its bands
	int nslots;    // slots per band row (a multiple of FS_AHEAD)
	int wc;        // carry words per band: w rounded up to FS_STEP
	int polls;     // FsRun::polls
};

// Scratch of a slab: nplanes channel planes, the carries of its bands, two
// edge rows per channel (carries into the slab and out of it, swapped from
// slab to slab) and the ticket counters.
struct FsScratch {
	uint4 *planes;       // [channel][band][slot][row]: 8 source values, then 8 quantized ones in the first half
	uint32_t *carry;     // [channel][band][wc]
	uint32_t *edge;      // [channel][2][wc]
	uint32_t *zeros;     // [FS_STEP * FS_ZERO_GROUPS]
	unsigned *tickets;   // [2]
	uint32_t *gave_up;   // FsRun::gave_up
};

// One channel's quantizer of v = u + 2048: q = clamp(floor(u * scale + bias),
// 0, maxv), error u - floor(q * deq - 2048).  shift 3: 12-bit v >> 7 against 4095 q / 31; shift 2: v >> 6,
// 65 q; shift 4: v >> 8, 273 q; one bit (shift 7): v >= 2048, 4095 q.  deq is
// exact or, for 4095 / 31, rounded up, so that the product's integer part is
// that of the integer division.
struct FsQuant {
	float scale, bias, maxv, deq;
};

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

__device__ __forceinline__ size_t fs_slot(const FsDims &d, int ch, int band, int j, int r)
{
	return (((size_t)ch * d.nb + band) * d.nslots + j) * FS_ROWS + r;
}

// 12-bit source value (s2tc_algorithm.cpp:1240) less 2048, as the bits of a
// half: an integer of at most 11 bits, which half holds exactly.
__device__ __forceinline__ uint32_t fs_src(uint32_t v)
{
	return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)((int)((v << 4) | (v >> 4)) - 2048));
}

// Source texels to channel planes ch0 .. ch0 + nch - 1 in wave order, empty
// carries, tickets and (first slab of the colour pass) zero edge rows.  One
// wave per slot.
__global__ __launch_bounds__(256) void k_fs_prepare(const uint8_t *__restrict__ src, int srccomps, FsDims d, int ch0,
                                                    int nch, FsScratch s, int zero_edges)
{
	const int r = (int)(threadIdx.x & 63), j = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), band = (int)blockIdx.y;
	if (j >= d.nslots) return;
	if (band == 0 && j == 0 && r < 2) s.tickets[r] = 0u;
	if (band == 0 && j == 0) s.zeros[r] = 0u;
	if (8 * j < d.wc && r < 8) {
		for (int c = ch0; c < ch0 + nch; ++c) s.carry[((size_t)c * d.nb + band) * d.wc + 8 * j + r] = NO_CARRY;
		if (band == 0 && zero_edges)
			for (int c = 0; c < 4; ++c) s.edge[(size_t)(2 * c) * d.wc + 8 * j + r] = 0u;
	}
	const int row = band * FS_ROWS + r, x0 = FS_STEP * j - 2 * r;
	if (row >= d.rows || x0 >= d.w || x0 + FS_STEP <= 0) return;  // never used as texels
	const size_t p0 = (size_t)(d.y0 + row) * (size_t)d.w;
	uint32_t tx[8];
	if (srccomps == 4 && x0 >= 0 && x0 + 8 <= d.w) {
		const u32x4_a4 *g = (const u32x4_a4 *)(src + (p0 + x0) * 4);
		const u32x4_a4 a = g[0], b = g[1];
#pragma unroll
		for (int i = 0; i < 4; ++i) {
			tx[i] = a[i];
			tx[4 + i] = b[i];
		}
	} else {
#pragma unroll
		for (int i = 0; i < 8; ++i) {
			const int x = x0 + i;
			tx[i] = 0;
			if (x < 0 || x >= d.w) continue;
			if (srccomps == 4) {
				tx[i] = ((const uint32_t *)src)[p0 + x];
			} else {
				const uint8_t *t = src + (p0 + x) * 3;
				tx[i] = (uint32_t)t[0] | ((uint32_t)t[1] << 8) | ((uint32_t)t[2] << 16);
			}
		}
	}
	for (int c = ch0; c < ch0 + nch; ++c) {
		uint32_t o[4];
#pragma unroll
		for (int i = 0; i < 4; ++i)
			o[i] = fs_src((tx[2 * i] >> (8 * c)) & 255u) | (fs_src((tx[2 * i + 1] >> (8 * c)) & 255u) << 16);
		s.planes[fs_slot(d, c, band, j, r)] = make_uint4(o[0], o[1], o[2], o[3]);
	}
}

// A lane's row state: the error to its right, A of the previous step and the
// downward sums that are not final yet.
struct FsRow {
	float right, fin, win1, win2;
};

// The stretches of a wave's steps: lanes still to start (texel x < 0), every
// lane inside the row, lanes past its end (x >= w), and both at once, which
// rows shorter than the lag have.
enum { FS_START = 1, FS_MAIN = 0, FS_END = 2, FS_BOTH = 3 };

// Eight steps from step t; lane2 = 2 r.  Texels outside the row make no error;
// the sums of the texels before them still drain.  The values u are the
// reference's less 2048, which the fmas of the quantizer add back.  21 VALU
// instructions a step; acc is dead unless the caller stores it.
template <int PHASE>
__device__ __forceinline__ void fs_steps(const uint4 &sv, const uint32_t (&c)[8], int t, int lane2, int w,
                                         const FsQuant &k, float one, FsRow &st, float (&fin)[8], float (&acc)[8], uint32_t (&q8)[2])
{
	const uint32_t sw[4] = {sv.x, sv.y, sv.z, sv.w};
	q8[0] = q8[1] = 0;
#pragma unroll
	for (int i = 0; i < 8; ++i) {
		// the row above, one lane down: its sum of the previous step (0 into lane 0)
		const float above = __builtin_bit_cast(
		    float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, st.fin), 0x138, 0xf, 0xf, true));
		const float a = (st.right + __builtin_bit_cast(float, c[i])) + above;
		acc[i] = a;
		const _Float16 src = __builtin_bit_cast(_Float16, (uint16_t)(sw[i >> 1] >> (16 * (i & 1))));
		const float u = __builtin_fmaf((float)src, one, a);  // one mixed-precision fma (one: an opaque 1)
		const float q = floorf(__builtin_amdgcn_fmed3f(__builtin_fmaf(u, k.scale, k.bias), 0.0f, k.maxv));
		float e = u - floorf(__builtin_fmaf(q, k.deq, -2048.0f));
		if (PHASE & FS_START) e = lane2 <= t + (i & ~1) ? e : 0.0f;  // lane2 is even
		if (PHASE & FS_END) e = lane2 > t + i - w ? e : 0.0f;
		q8[i >> 2] = __builtin_amdgcn_cvt_pk_u8_f32(q, (unsigned)(i & 3), q8[i >> 2]);
		// floyd (:1227-1233), C division: (7 e + 8) / 16, (3 e + 4) / 9, (5 e + 3) / 6
		const float e7 = truncf(__builtin_fmaf(e, 0.4375f, 0.5f));
		e -= e7;
		const float e3 = truncf(__builtin_fmaf(e, 0.333333343f, 0.444444448f));
		e -= e3;
		const float e5 = truncf(__builtin_fmaf(e, 0.833333373f, 0.5f));
		e -= e5;
		st.right = e7;
		st.fin = st.win1 + e3;
		st.win1 = st.win2 + e5;
		st.win2 = e;
		fin[i] = st.fin;
	}
}

typedef unsigned long long fs_pair;  // two carry words

// LDS of a workgroup of FS_WAVES waves: zeros for the lanes that get no
// carries, the ticket, then the carries of its bands but the last, wc words
// each.  Offsets count pairs.
extern __shared__ __align__(16) fs_pair fs_lds[];
#define FS_PAIRS (FS_STEP / 2)
#define FS_LDS_TICKET (FS_PAIRS * FS_ZERO_GROUPS)
#define FS_LDS_CARRY (FS_LDS_TICKET + FS_PAIRS)

// A group of eight carry words, from LDS (LOCAL) or memory.
struct FsGroup {
	uint32_t c[8];
	template <bool LOCAL> __device__ __forceinline__ void load(const fs_pair *p, int l, int group)
	{
#pragma unroll
		for (int i = 0; i < 4; ++i) {
			const fs_pair g = LOCAL ? __hip_atomic_load(fs_lds + l + (FS_PAIRS * group + i), __ATOMIC_RELAXED,
			                                            __HIP_MEMORY_SCOPE_WORKGROUP)
			                        : __hip_atomic_load(p + (FS_PAIRS * group + i), __ATOMIC_RELAXED,
			                                            __HIP_MEMORY_SCOPE_AGENT);
			c[2 * i] = (uint32_t)g;
			c[2 * i + 1] = (uint32_t)(g >> 32);
		}
	}
	__device__ __forceinline__ bool missing() const
	{
		uint32_t m = c[0];
#pragma unroll
		for (int i = 1; i < 8; ++i) m = max(m, c[i]);
		return m == NO_CARRY;
	}
	__device__ __forceinline__ void clear()
	{
#pragma unroll
		for (int i = 0; i < 8; ++i) c[i] = 0u;
	}
};

// What a wave's slots share.  The pointers move with the rounds of FS_AHEAD
// slots.
struct FsWave {
	int lane, lane2, w, ng;
	uint4 *P;              // slot j0 (this lane's words)
	const fs_pair *cin;    // lane 0: group j0 of the carries into the band; other lanes: zeros
	int lin;               // the same as an LDS offset
	int cstep;             // pairs from round to round in lane 0, else 0
	int outl;              // the lane that carries out: 63, in the last red band its last row, else none
	fs_pair *cout;         // group j0 - 16 of the carries out, to memory
	int lout;              // or to LDS at this offset
	bool red, rl_acc;      // the last red row: its read sums (even rows) or its downward ones
	FsQuant k;
	float one;
	FsRow st;
	float prev7;
	int patience;          // FsDims::polls, 0 after a wait that gave up
	uint32_t *gave_up;
};

// Slot u of the round at j0.  LIN, LOUT: the carries come from, go to LDS.  sv
// and g hold the slot's source values and carries and get those of a later
// one.  Loads past a band's last slot or group stay inside the scratch or the
// LDS (padded for them) and are not used.  A taken branch costs a lone wave
// about ten instructions, so the common path has none.
template <int PHASE, bool LIN, bool LOUT, int CA>
__device__ __forceinline__ void fs_slot_step(FsWave &f, int j0, int u, uint4 &sv, FsGroup &g)
{
	const int j = j0 + u;
	if (!(PHASE & FS_END) || j < f.ng) {
		if (__builtin_expect(__any((int)g.missing()), 0)) {
			// registers of its own, so that the common path waits for its
			// own prefetch alone
			FsGroup t;
			int left = f.patience * (LIN ? FS_LDS_POLLS : 1);
			bool miss;
			do {
				if (!LIN) __builtin_amdgcn_s_sleep(1);
				t.template load<LIN>(f.cin, f.lin, u);
				miss = __any((int)t.missing());
			} while (miss && --left > 0);
			if (__builtin_expect(miss, 0)) {
				t.clear();
				f.patience = 0;
				if (f.lane == 0) *f.gave_up = 1u;
			}
			g = t;
		}
	}
	float fin[8], acc[8];
	uint32_t q8[2];
	fs_steps<PHASE>(sv, g.c, FS_STEP * j, f.lane2, f.w, f.k, f.one, f.st, fin, acc, q8);
	// into the registers that are free now
	sv = f.P[(u + FS_AHEAD) * FS_ROWS];
	g.template load<LIN>(f.cin, f.lin, u + CA);
	*(uint2 *)&f.P[u * FS_ROWS] = make_uint2(q8[0], q8[1]);
	// lane 63's sums A[x], x = 8 j + i - FS_LAG, belong to texel x - 1 of the
	// row below: texels 8 m .. 8 m + 7 with the previous slot's last
	const int m = j - (FS_LAG + 2) / FS_STEP;
	if ((PHASE != FS_START || !LOUT) && f.lane == f.outl) {
		if (!LOUT && __builtin_expect(f.red, 0)) {
			uint32_t *rl = (uint32_t *)(f.cout - FS_PAIRS * (j0 - (FS_LAG + 2) / FS_STEP));
#pragma unroll
			for (int i = 0; i < 8; ++i) {
				const int x = FS_STEP * j + i - 2 * f.lane - (f.rl_acc ? 0 : 1);  // the alpha texel that reads it
				if (x >= 0 && x < f.w) rl[x] = __builtin_bit_cast(uint32_t, f.rl_acc ? acc[i] : fin[i]);
			}
		} else if (PHASE == FS_MAIN || (PHASE != FS_START && m >= 0 && m < f.ng)) {
			const float o[8] = {f.prev7, fin[0], fin[1], fin[2], fin[3], fin[4], fin[5], fin[6]};
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				const fs_pair v = (fs_pair)__builtin_bit_cast(uint32_t, o[2 * i]) |
				                  ((fs_pair)__builtin_bit_cast(uint32_t, o[2 * i + 1]) << 32);
				if (LOUT)
					__hip_atomic_store(fs_lds + f.lout + (FS_PAIRS * u + i), v, __ATOMIC_RELAXED,
					                   __HIP_MEMORY_SCOPE_WORKGROUP);
				else
					__hip_atomic_store(f.cout + (FS_PAIRS * u + i), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			}
		}
	}
	f.prev7 = fin[7];
}

template <int PHASE, bool LIN, bool LOUT, int CA>
__device__ __forceinline__ void fs_round(FsWave &f, int j0, uint4 (&sv)[FS_AHEAD], FsGroup (&g)[CA])
{
#pragma unroll
	for (int u = 0; u < FS_AHEAD; ++u) fs_slot_step<PHASE, LIN, LOUT, CA>(f, j0, u, sv[u], g[u % CA]);
	f.P += FS_AHEAD * FS_ROWS;
	if (LIN) f.lin += f.cstep;
	else f.cin += f.cstep;
	if (LOUT) f.lout += FS_AHEAD * FS_PAIRS;
	else f.cout += FS_AHEAD * FS_PAIRS;
}

// A wave's slots 0 .. nj - 1 in rounds (nslots is a multiple of FS_AHEAD),
// each stretch in a loop of its own so that the prefetched registers stay in
// place.
template <bool LIN, bool LOUT> __device__ __forceinline__ void fs_band(FsWave &f, int nj)
{
	constexpr int CA = LIN ? 1 : FS_AHEAD;
	uint4 sv[FS_AHEAD];
	FsGroup g[CA];
#pragma unroll
	for (int u = 0; u < FS_AHEAD; ++u) sv[u] = f.P[u * FS_ROWS];
#pragma unroll
	for (int u = 0; u < CA; ++u) g[u].template load<LIN>(f.cin, f.lin, u);
	int j0 = 0;
	if (f.w >= FS_LAG + 2) {
		for (; j0 < (FS_LAG + 2) / FS_STEP; j0 += FS_AHEAD) fs_round<FS_START, LIN, LOUT, CA>(f, j0, sv, g);
		for (; FS_STEP * (j0 + FS_AHEAD) <= f.w; j0 += FS_AHEAD) fs_round<FS_MAIN, LIN, LOUT, CA>(f, j0, sv, g);
		for (; j0 < nj; j0 += FS_AHEAD) fs_round<FS_END, LIN, LOUT, CA>(f, j0, sv, g);
	} else {
		for (; j0 < nj; j0 += FS_AHEAD) fs_round<FS_BOTH, LIN, LOUT, CA>(f, j0, sv, g);
	}
}

// The wavefront of one slab: one wave per (band, channel), WAVES consecutive
// bands per workgroup.  edge_in: which of the two edge rows carries into band
// 0; the last band carries out into the other (has_next: another slab
// follows).  last_red: channel 0 leaves what the alpha pass starts from in
// the alpha channel's edge row 0.
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void k_fs_rows(FsDims d, int ch0, int nch, FsQuant k0, FsQuant k1, FsQuant k2,
                                                        FsScratch s, int ticket, int edge_in, int has_next,
                                                        int last_red)
{
	FsWave f;
	f.lane = (int)(threadIdx.x & 63);
	const int wave = WAVES == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	unsigned id = 0;
	if constexpr (WAVES == 1) {
		if (f.lane == 0) id = atomicAdd(&s.tickets[ticket], 1u);
		id = (unsigned)__builtin_amdgcn_readfirstlane((int)id);
	} else {
		if (threadIdx.x == 0) fs_lds[FS_LDS_TICKET] = atomicAdd(&s.tickets[ticket], 1u);
		if (threadIdx.x < FS_LDS_TICKET) fs_lds[threadIdx.x] = 0u;
		for (int i = (int)threadIdx.x; i < (WAVES - 1) * d.wc / 2; i += 64 * WAVES) fs_lds[FS_LDS_CARRY + i] = ~0ull;
		__syncthreads();
		id = (unsigned)__builtin_amdgcn_readfirstlane((int)fs_lds[FS_LDS_TICKET]);
	}
	const int bg = (int)(id / (unsigned)nch), kc = (int)(id - (unsigned)bg * (unsigned)nch), ch = ch0 + kc;
	const int band = bg * WAVES + wave;
	if (band >= d.nb) return;
	const bool last_band = band == d.nb - 1;
	f.lane2 = 2 * f.lane;
	f.w = d.w;
	f.ng = d.wc / FS_STEP;
	f.k = kc == 0 ? k0 : kc == 1 ? k1 : k2;
	f.one = 1.0f;
	asm volatile("" : "+v"(f.one));
	const int lastrow = d.rows - 1 - band * FS_ROWS;  // lane of the slab's last row, in its last band
	f.red = last_red && last_band && ch == 0;
	f.rl_acc = ((d.y0 + d.rows - 1) & 1) == 0;
	f.P = s.planes + fs_slot(d, ch, band, 0, f.lane);
	f.cin = (const fs_pair *)(band == 0 ? s.edge + (size_t)(2 * ch + edge_in) * d.wc
	                                    : s.carry + ((size_t)ch * d.nb + band - 1) * d.wc);
	f.lin = FS_LDS_CARRY + (wave - 1) * (d.wc / 2);
	f.cstep = FS_AHEAD * FS_PAIRS;
	if (f.lane != 0) {
		f.cin = (const fs_pair *)s.zeros;
		f.lin = 0;
		f.cstep = 0;
	}
	const bool out = !last_band || has_next;
	f.outl = out ? FS_ROWS - 1 : f.red ? lastrow : -1;
	const int back = FS_PAIRS * ((FS_LAG + 2) / FS_STEP);  // group j0 - 16
	f.lout = FS_LDS_CARRY + wave * (d.wc / 2) - back;
	f.cout = (fs_pair *)(!last_band ? s.carry + ((size_t)ch * d.nb + band) * d.wc
	                                : s.edge + (size_t)(f.red ? 2 * 3 : 2 * ch + (edge_in ^ 1)) * d.wc) -
	         back;
	f.st = FsRow{0.0f, 0.0f, 0.0f, 0.0f};
	f.prev7 = 0.0f;
	f.patience = d.polls;
	f.gave_up = s.gave_up;
	// the band's last lane that matters does texel w (its sum drains) at this step
	const int nj = (d.w + (out ? FS_LAG + 1 : 2 * lastrow)) / FS_STEP + 1;
	if constexpr (WAVES == 1) {
		fs_band<false, false>(f, nj);
	} else {
		const bool lout = wave < WAVES - 1 && !last_band;
		if (wave == 0) {
			if (lout) fs_band<false, true>(f, nj);
			else fs_band<false, false>(f, nj);
		} else {
			if (lout) fs_band<true, true>(f, nj);
			else fs_band<true, false>(f, nj);
		}
	}
}

// Quantized planes to texels {r, g, b, a}.  alpha: -2 the planes hold alpha
// alone (only byte 3 is written), -1 from plane 3, -3 copied from the source,
// else the constant.
__global__ __launch_bounds__(256) void k_fs_finish(const uint8_t *__restrict__ src, FsDims d, FsScratch s, int alpha,
                                                   uint32_t *__restrict__ out)
{
	const int r = (int)(threadIdx.x & 63), j = (int)(blockIdx.x * 4 + (threadIdx.x >> 6)), band = (int)blockIdx.y;
	if (j >= d.nslots) return;
	const int row = band * FS_ROWS + r, x0 = FS_STEP * j - 2 * r;
	if (row >= d.rows || x0 >= d.w || x0 + FS_STEP <= 0) return;
	const size_t p0 = (size_t)(d.y0 + row) * (size_t)d.w;
	uint2 q[4];
#pragma unroll
	for (int c = 0; c < 4; ++c) {
		q[c] = make_uint2(0u, 0u);
		if (c < 3 ? alpha != -2 : alpha == -1 || alpha == -2) q[c] = *(const uint2 *)&s.planes[fs_slot(d, c, band, j, r)];
	}
	uint32_t t[8];
#pragma unroll
	for (int i = 0; i < 8; ++i) {
		const uint32_t sh = 8u * (i & 3);
		uint32_t b[4];
#pragma unroll
		for (int c = 0; c < 4; ++c) b[c] = ((i < 4 ? q[c].x : q[c].y) >> sh) & 255u;
		if (alpha >= 0) b[3] = (uint32_t)alpha;
		if (alpha == -3 && x0 + i >= 0 && x0 + i < d.w) b[3] = src[(p0 + x0 + i) * 4 + 3];
		t[i] = b[0] | (b[1] << 8) | (b[2] << 16) | (b[3] << 24);
	}
	if (alpha != -2 && x0 >= 0 && x0 + 8 <= d.w) {
		u32x4_a4 *g = (u32x4_a4 *)(out + p0 + x0);
		g[0] = u32x4_a4{t[0], t[1], t[2], t[3]};
		g[1] = u32x4_a4{t[4], t[5], t[6], t[7]};
		return;
	}
#pragma unroll
	for (int i = 0; i < 8; ++i) {
		const int x = x0 + i;
		if (x < 0 || x >= d.w) continue;
		if (alpha == -2) ((uint8_t *)(out + p0 + x))[3] = (uint8_t)(t[i] >> 24);
		else out[p0 + x] = t[i];
	}
}

// The whole dither of up to FS_SMALL texels, one lane per channel, the alpha lane
// after the others: its first row starts from what the red lane left.  Bound:
// launches, then a serial chain of some forty instructions a texel.  Measured
// (MI355X, rgb565_image, one alpha bit; four launches of the wavefront -> one):
// 1 x 1 37.7 -> 25.9 us, 4 x 4 38.7 -> 30.4, 6 x 6 38.8 -> 36.2, 7 x 7 39.5 -> 39.9,
// 8 x 8 39.2 -> 44.0.
#define FS_SMALL 36

__global__ __launch_bounds__(64) void k_fs_small(const uint8_t *__restrict__ src, int srccomps, int w, int h, int nch,
                                                 FsQuant k0, FsQuant k1, FsQuant k2, FsQuant k3, int alpha,
                                                 uint32_t *__restrict__ out)
{
	__shared__ uint32_t tex[FS_SMALL];
	__shared__ uint8_t level[4][FS_SMALL];
	__shared__ float down[4][FS_SMALL + 2];  // A of the next row, in place
	const int t = (int)threadIdx.x, n = w * h;
	if (t < n) {
		if (srccomps == 4) tex[t] = ((const uint32_t *)src)[t];
		else tex[t] = (uint32_t)src[3 * t] | ((uint32_t)src[3 * t + 1] << 8) | ((uint32_t)src[3 * t + 2] << 16);
	}
	for (int i = t; i < 4 * (FS_SMALL + 2); i += 64) (&down[0][0])[i] = 0.0f;
	__syncthreads();
	const FsQuant k = t == 0 ? k0 : t == 1 ? k1 : t == 2 ? k2 : k3;
	for (int pass = 0; pass < 2; ++pass) {
		if (pass == 0 ? t < 3 : t == 3 && nch == 4) {
			for (int y = 0; y < h; ++y) {
				float right = 0.0f, win1 = 0.0f, win2 = 0.0f;
				for (int x = 0; x <= w; ++x) {
					float e = 0.0f;
					if (x < w) {
						const float a = right + down[t][x + 1];
						const uint32_t v = (tex[y * w + x] >> (8 * t)) & 255u;
						const float u = a + (float)((int)((v << 4) | (v >> 4)) - 2048);
						const float q = floorf(__builtin_amdgcn_fmed3f(__builtin_fmaf(u, k.scale, k.bias), 0.0f, k.maxv));
						e = u - floorf(__builtin_fmaf(q, k.deq, -2048.0f));
						level[t][y * w + x] = (uint8_t)q;
						if (t == 0 && y == h - 1 && !(y & 1)) down[3][x + 1] = a;
					}
					const float e7 = truncf(__builtin_fmaf(e, 0.4375f, 0.5f));
					e -= e7;
					const float e3 = truncf(__builtin_fmaf(e, 0.333333343f, 0.444444448f));
					e -= e3;
					const float e5 = truncf(__builtin_fmaf(e, 0.833333373f, 0.5f));
					e -= e5;
					right = e7;
					const float fin = win1 + e3;
					down[t][x] = fin;
					if (t == 0 && y == h - 1 && (y & 1) && x > 0) down[3][x] = fin;
					win1 = win2 + e5;
					win2 = e;
				}
			}
		}
		__syncthreads();
	}
	if (t < n) {
		const uint32_t a = nch == 4 ? level[3][t] : alpha >= 0 ? (uint32_t)alpha : tex[t] >> 24;
		out[t] = (uint32_t)level[0][t] | ((uint32_t)level[1][t] << 8) | ((uint32_t)level[2][t] << 16) | (a << 24);
	}
}

// ---- host ----

// LDS bytes of a workgroup of FS_WAVES waves for rows of wc carry words, and the
// widest rows whose carries fit.
static constexpr size_t fs_lds_bytes(int wc)
{
	return (size_t)FS_LDS_CARRY * 8 + ((size_t)(FS_WAVES - 1) * wc + FS_PAD_WORDS) * 4;
}
#define FS_LDS_WIDTH 13216
static_assert(fs_lds_bytes(FS_LDS_WIDTH) <= FS_LDS_MAX && fs_lds_bytes(FS_LDS_WIDTH + FS_STEP) > FS_LDS_MAX,
              "FS_LDS_WIDTH");

// The image is dithered in slabs of whole bands whose planes fit FsRun::slab;
// the wavefront drains between slabs, which a 4096-wide image does every 15,000
// rows with FS_SLAB.
static FsDims fs_dims(int w, int h, size_t slab)
{
	FsDims d{};
	d.w = w;
	d.wc = (w + FS_STEP - 1) / FS_STEP * FS_STEP;
	d.nslots = d.wc / FS_STEP + (FS_LAG + 2) / FS_STEP;
	d.nslots = (d.nslots + FS_AHEAD - 1) / FS_AHEAD * FS_AHEAD;
	const size_t band = (size_t)4 * d.nslots * FS_ROWS * sizeof(uint4);
	const long long cap = std::max<long long>(1, (long long)(slab / band));
	d.nb = (int)std::min<long long>(((long long)h + FS_ROWS - 1) / FS_ROWS, cap);
	return d;
}

static size_t fs_align(size_t n) { return (n + 255) & ~(size_t)255; }
static size_t fs_plane_bytes(const FsDims &d)
{
	return fs_align(((size_t)4 * d.nb * d.nslots + FS_AHEAD) * FS_ROWS * sizeof(uint4));
}
static size_t fs_carry_bytes(const FsDims &d) { return fs_align(((size_t)4 * d.nb * d.wc + FS_PAD_WORDS) * 4); }
static size_t fs_edge_bytes(const FsDims &d) { return fs_align(((size_t)8 * d.wc + FS_PAD_WORDS) * 4); }

size_t rgb565_fs_scratch_bytes(int w, int h, size_t slab)
{
	const FsDims d = fs_dims(w, h, slab);
	return fs_plane_bytes(d) + fs_carry_bytes(d) + fs_edge_bytes(d) + 512;
}

static FsQuant fs_quant(int shift)
{
	const int maxval = (1 << (8 - shift)) - 1;
	float deq = (float)(4095.0 / maxval);
	if ((double)deq < 4095.0 / maxval) deq = std::nextafter(deq, 8192.0f);
	const float scale = 1.0f / (float)(1 << (shift + 4));
	return FsQuant{scale, 2048.0f * scale, (float)maxval, deq};
}

static int fs_rows(const FsDims &d, int ch0, int nch, FsQuant k0, FsQuant k1, FsQuant k2, const FsScratch &s,
                   int ticket, int edge_in, int has_next, int last_red, hipStream_t st)
{
	const size_t lds = fs_lds_bytes(d.wc);
	if (d.wc > FS_LDS_WIDTH) {
		k_fs_rows<1><<<(unsigned)(d.nb * nch), 64, 0, st>>>(d, ch0, nch, k0, k1, k2, s, ticket, edge_in, has_next,
		                                                    last_red);
	} else {
		if (lds > 65536)
			if (int r = hip_check(hipFuncSetAttribute((const void *)k_fs_rows<FS_WAVES>,
			                                          hipFuncAttributeMaxDynamicSharedMemorySize, FS_LDS_MAX),
			                      "hipFuncSetAttribute"))
				return r;
		const unsigned groups = (unsigned)((d.nb + FS_WAVES - 1) / FS_WAVES);
		k_fs_rows<FS_WAVES><<<groups * nch, 64 * FS_WAVES, lds, st>>>(d, ch0, nch, k0, k1, k2, s, ticket, edge_in,
		                                                              has_next, last_red);
	}
	return hip_check(hipGetLastError(), "dither FS wavefront");
}

int launch_rgb565_fs(const uint8_t *src, int srccomps, int w, int h, int alphabits, uint8_t *out, void *d_scratch,
                     hipStream_t st, const FsRun &run)
{
	if (!run.gave_up) return set_error(S2TC_E_ARG, "the Floyd-Steinberg dither needs a word for its waits");
	FsDims full = fs_dims(w, h, run.slab);
	full.polls = (int)std::min(run.polls, FS_POLLS);
	FsScratch s;
	s.gave_up = run.gave_up;
	uint8_t *p = (uint8_t *)d_scratch;
	s.planes = (uint4 *)p;
	p += fs_plane_bytes(full);
	s.carry = (uint32_t *)p;
	p += fs_carry_bytes(full);
	s.edge = (uint32_t *)p;
	p += fs_edge_bytes(full);
	s.zeros = (uint32_t *)p;
	s.tickets = (unsigned *)p + FS_STEP * FS_ZERO_GROUPS;
	const bool alpha_fs = srccomps == 4 && (alphabits == 1 || alphabits == 4);
	const FsQuant q5 = fs_quant(3), q6 = fs_quant(2), qa = fs_quant(alphabits == 1 ? 7 : 4);
	const int slab_rows = full.nb * FS_ROWS;
	const bool one_slab = slab_rows >= h;
	const int plain_alpha = srccomps == 4 ? -3 : (1 << alphabits) - 1;
	if ((long long)w * h <= FS_SMALL) {
		k_fs_small<<<1, 64, 0, st>>>(src, srccomps, w, h, alpha_fs ? 4 : 3, q5, q6, q5, qa, plain_alpha, (uint32_t *)out);
		return hip_check(hipGetLastError(), "dither FS kernel");
	}
	// colour, then alpha from the errors that red left: all in one round of
	// kernels where the image is one slab, else colour slabs, then alpha slabs
	for (int pass = 0; pass < (alpha_fs && !one_slab ? 2 : 1); ++pass) {
		const int ch0 = pass ? 3 : 0, nch = pass ? 1 : alpha_fs && one_slab ? 4 : 3;
		int edge_in = 0;
		for (int y0 = 0; y0 < h; y0 += slab_rows, edge_in ^= 1) {
			FsDims d = full;
			d.y0 = y0;
			d.rows = std::min(slab_rows, h - y0);
			d.nb = (d.rows + FS_ROWS - 1) / FS_ROWS;
			const int has_next = y0 + d.rows < h ? 1 : 0;
			const dim3 grid((unsigned)((d.nslots + 3) / 4), (unsigned)d.nb);
			k_fs_prepare<<<grid, 256, 0, st>>>(src, srccomps, d, ch0, nch, s, pass == 0 && y0 == 0 ? 1 : 0);
			if (pass == 0)
				if (int r = fs_rows(d, 0, 3, q5, q6, q5, s, 0, edge_in, has_next, alpha_fs && !has_next ? 1 : 0, st))
					return r;
			if (pass == 1 || nch == 4)
				if (int r = fs_rows(d, 3, 1, qa, qa, qa, s, 1, edge_in, has_next, 0, st)) return r;
			const int alpha = pass ? -2 : nch == 4 ? -1 : alpha_fs ? 0 : plain_alpha;
			k_fs_finish<<<grid, 256, 0, st>>>(src, d, s, alpha, (uint32_t *)out);
			if (int r = hip_check(hipGetLastError(), "dither FS kernels")) return r;
		}
	}
	return 0;
}

}  // namespace s2tc
