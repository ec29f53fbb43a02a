// dither.hip - rgb565_image on the GPU (s2tc_algorithm.cpp:1196-1465).
//
// DITHER_NONE is a per-texel shift (k_quantize_none).
//
// DITHER_SIMPLE carries one running error per channel through the whole
// image in row-major order (:1307-1349).  The error is a small finite state:
// diffuse() with shift s keeps d in [-(2^s - 1), 2^s - 1] (15 states for
// shift 3, 7 for shift 2, 31 for shift 4), and diffuse1() keeps
// e = d + 127 = (127 + sum of inputs) mod 255.  The chain is a scan over
// transition maps: a lane finds the map of its chunk of L texels, a wave
// scans the maps of its 64 chunks, the waves' maps are scanned in turn, and
// every lane then re-runs its chunk from its start state.
//
// A map is one byte per start state, d + 2^s, four states to a register,
// and a texel moves all of them at once (SimpleMap::step): with v = 2^s q + m
// and t = m + d, the quantizer's floor is q + fl for fl = floor(t / 2^s) in
// {-1, 0, 1}, and the new d is t mod 2^s less a value that depends on q and fl
// alone, which is one byte permute of a table entry for v.  So the 37 states
// of r, g and b take 60 instructions a texel, where one lane per state took
// three waves' worth of lanes at about ten instructions each.
//
// Kernels: k_simple_maps (maps of chunks and waves), k_simple_states (start
// state of every wave; only above 64 waves, else each wave scans them by
// itself), k_simple_emit.  Up to SIMPLE_ONE texels one workgroup does it all
// in one launch (k_simple_one).  Texels go through LDS both ways, so memory
// sees whole lines while each lane works on its own chunk.
//
// Bound: instruction issue (about 75 per texel for the maps, 30 for the
// second run) over 12 bytes a texel; on small images the latency of the
// kernels' loads.  The loops are short (4 texels), as a chain of cold
// instruction lines costs small images more than the loop's branches.
// Measured (MI355X): a 4096 x 1024 RGBA band takes 18 + 6 + 10 us; with one
// lane per state and byte stores it was 104 + 16 + 18 + 90 us and a fifth
// kernel for the alpha.  256 x 256: 10 + 6 us (was 38 us in four kernels),
// 20 x 12: 7 us (16 us).
//
// DITHER_FLOYDSTEINBERG is in dither_fs.hip.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "s2tc_internal.h"

namespace s2tc {

#define SIMPLE_WG 256        // lanes of a workgroup, one chunk each
#define SIMPLE_ONE_LSH 3     // k_simple_one: texels per chunk (logarithm)
#define SIMPLE_ONE (1024 << SIMPLE_ONE_LSH)

__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel)
{
	return __builtin_amdgcn_perm(hi, lo, sel);
}

// Transition map of a diffuse(SH) channel: byte i of the ND registers is the
// end state (d + OFF, at least 1) from start state i.
template <int SH> struct SimpleMap {
	static constexpr int OFF = 1 << SH;
	static constexpr int ND = SH == 2 ? 2 : SH == 3 ? 4 : 8;
	uint32_t d[ND];

	__device__ __forceinline__ void identity()
	{
#pragma unroll
		for (int i = 0; i < ND; ++i) d[i] = 0x03020100u + 0x04040404u * (uint32_t)i;
	}
	// The table entry of source value v: bytes 0..2 are OFF - E[fl] for fl =
	// -1, 0, 1, byte 3 is m.  E = r >> (8 - 2 SH) for the level r = q + fl; a
	// level below 0 or above the last one is clamped, which leaves d = t (E =
	// OFF) or d = t - OFF + 1 (E = -1).
	static constexpr uint32_t entry(uint32_t v)
	{
		const int q = (int)(v >> SH), m = (int)(v & (uint32_t)(OFF - 1)), last = (1 << (8 - SH)) - 1, s = 8 - 2 * SH;
		const int e0 = q == 0 ? OFF : (q - 1) >> s, e1 = q >> s, e2 = q == last ? -1 : (q + 1) >> s;
		return (uint32_t)(OFF - e0) | ((uint32_t)(OFF - e1) << 8) | ((uint32_t)(OFF - e2) << 16) | ((uint32_t)m << 24);
	}
	// one texel: byte x = t + OFF = (d + OFF) + m < 2^6, and the sums stay
	// below 2 OFF, so the bytes never carry into each other
	__device__ __forceinline__ void step(uint32_t k)
	{
		const uint32_t m = perm(k, k, 0x03030303u);
#pragma unroll
		for (int i = 0; i < ND; ++i) {
			const uint32_t x = d[i] + m;
			d[i] = (x & (0x01010101u * (uint32_t)(OFF - 1))) + perm(k, k, (x >> SH) & 0x03030303u);
		}
	}
	// d[] as a table of 16 bytes at t
	static __device__ __forceinline__ uint32_t look16(const uint32_t *t, uint32_t sel)
	{
		const uint32_t lo = sel & 0x07070707u;
		return perm(perm(t[3], t[2], lo), perm(t[1], t[0], lo), ((sel >> 1) & 0x04040404u) | 0x03020100u);
	}
	// four lookups (selectors below the number of states)
	__device__ __forceinline__ uint32_t look(uint32_t sel) const
	{
		if constexpr (ND == 2) return perm(d[1], d[0], sel);
		else if constexpr (ND == 4) return look16(d, sel);
		else {
			const uint32_t s = sel & 0x0f0f0f0fu;
			return perm(look16(d + 4, s), look16(d, s), ((sel >> 2) & 0x04040404u) | 0x03020100u);
		}
	}
	__device__ __forceinline__ uint32_t at(uint32_t state) const { return look(state) & 255u; }
	// this map after `first`
	__device__ __forceinline__ void after(const SimpleMap &first)
	{
		uint32_t o[ND];
#pragma unroll
		for (int i = 0; i < ND; ++i) o[i] = look(first.d[i]);
#pragma unroll
		for (int i = 0; i < ND; ++i) d[i] = o[i];
	}
};

// The mod-255 channel (diffuse1): a chunk adds its sum to the state.
struct SimpleSum {
	static constexpr int ND = 1;
	uint32_t d[1];
	__device__ __forceinline__ void identity() { d[0] = 0u; }
	__device__ __forceinline__ uint32_t at(uint32_t state) const { return (state + d[0]) % 255u; }
	__device__ __forceinline__ void after(const SimpleSum &first) { d[0] = (d[0] + first.d[0]) % 255u; }
};

// no dithered alpha
struct SimpleNone {
	static constexpr int ND = 0;
	uint32_t d[1];
	__device__ __forceinline__ void identity() {}
	__device__ __forceinline__ uint32_t at(uint32_t) const { return 0u; }
	__device__ __forceinline__ void after(const SimpleNone &) {}
};

// The map of the lane that DPP control CTRL names, the identity in lanes that
// have none (or whose row is not in ROWS).
template <int CTRL, int ROWS, class M> __device__ __forceinline__ M dpp_map(const M &m)
{
	M r;
	r.identity();
#pragma unroll
	for (int i = 0; i < M::ND; ++i)
		r.d[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)r.d[i], (int)m.d[i], CTRL, ROWS, 0xf, false);
	return r;
}
// Inclusive scan over the 64 lanes of a wave, lane 0 first: row_shr 1, 2, 4,
// 8 inside the rows of 16, then lane 15 of rows 0 and 2 to the next row and
// lane 31 to the upper half (row_bcast 15, 31).
template <class M> __device__ __forceinline__ void wave_scan(M &m)
{
	m.after(dpp_map<0x111, 0xf>(m));
	m.after(dpp_map<0x112, 0xf>(m));
	m.after(dpp_map<0x114, 0xf>(m));
	m.after(dpp_map<0x118, 0xf>(m));
	m.after(dpp_map<0x142, 0xa>(m));
	m.after(dpp_map<0x143, 0xc>(m));
}
template <class M> __device__ __forceinline__ M exclusive(const M &m) { return dpp_map<0x138, 0xf>(m); }  // wave_shr:1

// ALPHA kinds of a call
enum { ALPHA_PLAIN = 0, ALPHA_MOD = 1, ALPHA_4 = 2 };
template <int ALPHA> struct AlphaMap { typedef SimpleNone T; };
template <> struct AlphaMap<ALPHA_MOD> { typedef SimpleSum T; };
template <> struct AlphaMap<ALPHA_4> { typedef SimpleMap<4> T; };

template <int ALPHA> struct Maps {
	SimpleMap<3> r, b;
	SimpleMap<2> g;
	typename AlphaMap<ALPHA>::T a;
	__device__ __forceinline__ void identity()
	{
		r.identity();
		g.identity();
		b.identity();
		a.identity();
	}
};

// The start states of the reference: d = 0 (r, g, b, 4-bit alpha), e = 127.
__device__ __forceinline__ uint32_t start_states(int alpha)
{
	return 8u | (4u << 8) | (8u << 16) | ((alpha == ALPHA_MOD ? 127u : 16u) << 24);
}

// Scratch: maps of every chunk (exclusive within its wave), of every wave,
// and every wave's start states {r, g, b, a}.  Registers of a map are stored
// together, per channel.
struct SimpleScratch {
	uint32_t *r, *g, *b, *a;      // [chunk][ND]
	uint32_t *wr, *wg, *wb, *wa;  // [wave][ND]
	uint32_t *ws;                 // [wave]
	long long nw;                 // waves
};

template <class M> __device__ __forceinline__ void store_map(uint32_t *p, long long i, const M &m)
{
	if constexpr (M::ND == 1) p[i] = m.d[0];
	else if constexpr (M::ND == 2) *(uint2 *)(p + 2 * i) = make_uint2(m.d[0], m.d[1]);
	else if constexpr (M::ND >= 4)
#pragma unroll
		for (int k = 0; k < M::ND / 4; ++k)
			*(uint4 *)(p + M::ND * i + 4 * k) = make_uint4(m.d[4 * k], m.d[4 * k + 1], m.d[4 * k + 2], m.d[4 * k + 3]);
}
template <class M> __device__ __forceinline__ void load_map(const uint32_t *p, long long i, M &m)
{
#pragma unroll
	for (int k = 0; k < M::ND; ++k) m.d[k] = p[M::ND * i + k];
}

// A workgroup's LDS: the tables of the maps, then one word per texel, chunk
// after chunk with a gap of one word, so that the lanes of a wave start in
// different banks.  The chunk length is 1 << lsh.
extern __shared__ __align__(16) uint32_t simple_lds[];

struct EntryTables {
	uint32_t t[768];  // 256 entries each for shift 3, 2 and 4
};
static constexpr EntryTables entry_tables()
{
	EntryTables e{};
	for (unsigned v = 0; v < 256; ++v) {
		e.t[v] = SimpleMap<3>::entry(v);
		e.t[256 + v] = SimpleMap<2>::entry(v);
		e.t[512 + v] = SimpleMap<4>::entry(v);
	}
	return e;
}
static __device__ const EntryTables c_entries = entry_tables();

template <int ALPHA> constexpr int table_words() { return ALPHA == ALPHA_4 ? 768 : 512; }

// The workgroup's cnt texels from src as words {r, g, b, a} (a = 0 for three
// components); the words past them, up to `room`, are 0.
template <int COMPS>
__device__ __forceinline__ void load_texels(const uint8_t *src, int cnt, int room, int lsh, uint32_t *tex)
{
	const uint32_t *g = (const uint32_t *)src;
	for (int q = (int)threadIdx.x; 4 * q < room; q += (int)blockDim.x) {
		uint32_t t[4];
		if (4 * q + 4 <= cnt) {
			if constexpr (COMPS == 4) {
				const uint4 v = ((const uint4 *)g)[q];
				t[0] = v.x;
				t[1] = v.y;
				t[2] = v.z;
				t[3] = v.w;
			} else {
				const uint32_t a = g[3 * q], b = g[3 * q + 1], c = g[3 * q + 2];
				t[0] = a & 0xffffffu;
				t[1] = (a >> 24) | ((b & 0xffffu) << 8);
				t[2] = (b >> 16) | ((c & 0xffu) << 16);
				t[3] = c >> 8;
			}
		} else {
#pragma unroll
			for (int k = 0; k < 4; ++k) {
				const int i = 4 * q + k;
				t[k] = 0;
				if (i < cnt && COMPS == 4) t[k] = g[i];
				if (i < cnt && COMPS == 3)
					t[k] = (uint32_t)src[3 * i] | ((uint32_t)src[3 * i + 1] << 8) | ((uint32_t)src[3 * i + 2] << 16);
			}
		}
		const int at = 4 * q + ((4 * q) >> lsh);
#pragma unroll
		for (int k = 0; k < 4; ++k) tex[at + k] = t[k];
	}
}

// The maps of the lane's chunk: cnt of its words (a multiple of 4 unless the
// image ends in it).
template <int ALPHA>
__device__ __forceinline__ void chunk_maps(const uint32_t *tex, int cnt, const uint32_t *tab, Maps<ALPHA> &m)
{
	m.identity();
	const auto step = [&](uint32_t t) {
		m.r.step(tab[t & 255u]);
		m.g.step(tab[256 + ((t >> 8) & 255u)]);
		m.b.step(tab[(t >> 16) & 255u]);
		if constexpr (ALPHA == ALPHA_4) m.a.step(tab[512 + (t >> 24)]);
		if constexpr (ALPHA == ALPHA_MOD) m.a.d[0] += t >> 24;
	};
	int i = 0;
	for (; i + 4 <= cnt; i += 4) {
		uint32_t t[4];
#pragma unroll
		for (int k = 0; k < 4; ++k) t[k] = tex[i + k];
#pragma unroll
		for (int k = 0; k < 4; ++k) step(t[k]);
	}
	for (; i < cnt; ++i) step(tex[i]);
	if constexpr (ALPHA == ALPHA_MOD) m.a.d[0] %= 255u;
}

// One texel of diffuse(SH): d becomes the new error, returns the level.
template <int SH> __device__ __forceinline__ uint32_t diffuse(int &d, uint32_t v)
{
	const int s = (int)v + d;
	const int r = min(max(s >> SH, 0), (1 << (8 - SH)) - 1);
	d = s - ((r << SH) | (r >> (8 - 2 * SH)));
	return (uint32_t)r;
}

// Re-runs the lane's chunk of `len` words (a multiple of 4) from its states
// {r, g, b, a}, in place.  plain: the alpha byte where none is dithered (-1:
// the source's).
template <int ALPHA>
__device__ __forceinline__ void emit_chunk(uint32_t *tex, int len, uint32_t states, int plain)
{
	int dr = (int)(states & 255u) - 8, dg = (int)((states >> 8) & 255u) - 4, db = (int)((states >> 16) & 255u) - 8;
	int da = (int)(states >> 24) - (ALPHA == ALPHA_4 ? 16 : 0);
	const uint32_t keep = plain < 0 ? 0xff000000u : 0u, add = plain < 0 ? 0u : (uint32_t)plain << 24;
	for (int i = 0; i < len; i += 4) {
		uint32_t t[4];
#pragma unroll
		for (int k = 0; k < 4; ++k) t[k] = tex[i + k];
#pragma unroll
		for (int k = 0; k < 4; ++k) {
			uint32_t o = diffuse<3>(dr, t[k] & 255u);
			o |= diffuse<2>(dg, (t[k] >> 8) & 255u) << 8;
			o |= diffuse<3>(db, (t[k] >> 16) & 255u) << 16;
			if constexpr (ALPHA == ALPHA_4) {
				o |= diffuse<4>(da, t[k] >> 24) << 24;
			} else if constexpr (ALPHA == ALPHA_MOD) {
				const int s = da + (int)(t[k] >> 24);  // d + src >= 128 with e = d + 127
				o |= s >= 255 ? 1u << 24 : 0u;
				da = s >= 255 ? s - 255 : s;
			} else {
				o |= (t[k] & keep) | add;
			}
			t[k] = o;
		}
#pragma unroll
		for (int k = 0; k < 4; ++k) tex[i + k] = t[k];
	}
}

// The workgroup's first cnt words to out.
__device__ __forceinline__ void store_texels(const uint32_t *tex, int cnt, int lsh, uint32_t *out)
{
	for (int i = (int)threadIdx.x; i < cnt; i += (int)blockDim.x) out[i] = tex[i + (i >> lsh)];
}

// Maps of the workgroup's chunks and waves.  raw (may be null): takes the
// texels as words.
template <int COMPS, int ALPHA>
__global__ __launch_bounds__(SIMPLE_WG) void k_simple_maps(const uint8_t *__restrict__ src, long long n, int lsh,
                                                           SimpleScratch s, uint32_t *__restrict__ raw)
{
	uint32_t *tab = simple_lds, *tex = simple_lds + table_words<ALPHA>();
	const int L = 1 << lsh;
	const long long p0 = (long long)blockIdx.x * SIMPLE_WG << lsh, chunk = (long long)blockIdx.x * SIMPLE_WG + threadIdx.x;
	const int cnt = (int)min((long long)SIMPLE_WG << lsh, n - p0);
	for (int i = (int)threadIdx.x; i < table_words<ALPHA>(); i += SIMPLE_WG) tab[i] = c_entries.t[i];
	load_texels<COMPS>(src + p0 * COMPS, cnt, SIMPLE_WG << lsh, lsh, tex);
	__syncthreads();
	if (raw) store_texels(tex, cnt, lsh, raw + p0);
	Maps<ALPHA> m;
	chunk_maps<ALPHA>(tex + (int)threadIdx.x * (L + 1), min(L, max(0, cnt - ((int)threadIdx.x << lsh))), tab, m);
	wave_scan(m.r);
	wave_scan(m.g);
	wave_scan(m.b);
	wave_scan(m.a);
	const long long wave = chunk >> 6;
	if (wave >= s.nw) return;
	if ((threadIdx.x & 63) == 63) {
		store_map(s.wr, wave, m.r);
		store_map(s.wg, wave, m.g);
		store_map(s.wb, wave, m.b);
		store_map(s.wa, wave, m.a);
	}
	store_map(s.r, chunk, exclusive(m.r));
	store_map(s.g, chunk, exclusive(m.g));
	store_map(s.b, chunk, exclusive(m.b));
	store_map(s.a, chunk, exclusive(m.a));
}

// Start states of the waves of one channel (blockIdx.x): each thread composes
// a run of consecutive maps, the workgroup scans those, and each thread then
// walks its run.  carry_in / carry_out: the error states before and after the
// texels (null: the reference's initial ones).
template <class M>
__device__ __forceinline__ void scan_states(const uint32_t *maps, long long nw, int ch, uint32_t init, uint8_t *ws,
                                            uint8_t *carry_out, uint32_t *lds)
{
	const int tid = (int)threadIdx.x, lane = tid & 63, wv = tid >> 6;
	const long long per = (nw + 1023) / 1024, lo = min(nw, per * tid), hi = min(nw, lo + per);
	M m;
	m.identity();
	for (long long i = lo; i < hi; ++i) {
		M e;
		load_map(maps, i, e);
		e.after(m);
		m = e;
	}
	wave_scan(m);
	if (lane == 63)
#pragma unroll
		for (int k = 0; k < M::ND; ++k) lds[wv * M::ND + k] = m.d[k];
	__syncthreads();
	M t;  // the 16 waves' maps, scanned by lanes 0..15 of every wave
	t.identity();
	if (lane < 16) load_map(lds, lane, t);
	wave_scan(t);
	const uint32_t after = t.at(init);  // lane w: the state after wave w
	const uint32_t before = (uint32_t)__shfl((int)after, max(wv - 1, 0), 64);
	uint32_t st = exclusive(m).at(wv ? before : init);
	for (long long i = lo; i < hi; ++i) {
		M e;
		load_map(maps, i, e);
		ws[4 * i + ch] = (uint8_t)st;
		st = e.at(st);
	}
	if (carry_out && tid == 1023) carry_out[ch] = (uint8_t)st;
}

template <int ALPHA>
__global__ __launch_bounds__(1024) void k_simple_states(SimpleScratch s, const uint8_t *__restrict__ carry_in,
                                                        uint8_t *__restrict__ carry_out)
{
	__shared__ uint32_t lds[16 * 8];
	const int ch = (int)blockIdx.x;
	const uint32_t init = carry_in ? carry_in[ch] : (start_states(ALPHA) >> (8 * ch)) & 255u;
	uint8_t *ws = (uint8_t *)s.ws;
	if (ch == 0) scan_states<SimpleMap<3>>(s.wr, s.nw, 0, init, ws, carry_out, lds);
	else if (ch == 1) scan_states<SimpleMap<2>>(s.wg, s.nw, 1, init, ws, carry_out, lds);
	else if (ch == 2) scan_states<SimpleMap<3>>(s.wb, s.nw, 2, init, ws, carry_out, lds);
	else if constexpr (ALPHA != ALPHA_PLAIN)
		scan_states<typename AlphaMap<ALPHA>::T>(s.wa, s.nw, 3, init, ws, carry_out, lds);
}

// The start state of wave `wave` and the state after all nw <= 64 waves, by a
// scan of the waves' maps over the lanes.
template <class M>
__device__ __forceinline__ uint32_t scan_here(const uint32_t *maps, int nw, int wave, uint32_t init, int lane,
                                              uint32_t &last)
{
	if constexpr (M::ND == 0) {
		last = 0;
		return 0;
	} else {
		M m;
		m.identity();
		if (lane < nw) load_map(maps, lane, m);
		wave_scan(m);
		const uint32_t v = m.at(init);
		last = (uint32_t)__shfl((int)v, nw - 1, 64);
		const uint32_t before = (uint32_t)__shfl((int)v, max(wave - 1, 0), 64);
		return wave ? before : init;
	}
}

// src may be out: a workgroup has read its texels before it writes them.
template <int COMPS, int ALPHA>
__global__ __launch_bounds__(SIMPLE_WG) void k_simple_emit(const uint8_t *src, long long n, int lsh, int plain,
                                                           SimpleScratch s, int scan,
                                                           const uint8_t *__restrict__ carry_in,
                                                           uint8_t *__restrict__ carry_out, uint32_t *out)
{
	uint32_t *tex = simple_lds;
	const int lane = (int)(threadIdx.x & 63), L = 1 << lsh;
	const long long p0 = (long long)blockIdx.x * SIMPLE_WG << lsh, chunk = (long long)blockIdx.x * SIMPLE_WG + threadIdx.x;
	const long long wave = min(chunk >> 6, s.nw - 1);  // waves past the end have no texels
	const int cnt = (int)min((long long)SIMPLE_WG << lsh, n - p0);
	load_texels<COMPS>(src + p0 * COMPS, cnt, SIMPLE_WG << lsh, lsh, tex);
	uint32_t ws;
	if (scan) {
		uint32_t init = start_states(ALPHA);
		if (carry_in) init = *(const uint32_t *)carry_in;
		const int nw = (int)s.nw, w = (int)wave;
		uint32_t e0, e1, e2, e3;
		ws = scan_here<SimpleMap<3>>(s.wr, nw, w, init & 255u, lane, e0);
		ws |= scan_here<SimpleMap<2>>(s.wg, nw, w, (init >> 8) & 255u, lane, e1) << 8;
		ws |= scan_here<SimpleMap<3>>(s.wb, nw, w, (init >> 16) & 255u, lane, e2) << 16;
		ws |= scan_here<typename AlphaMap<ALPHA>::T>(s.wa, nw, w, init >> 24, lane, e3) << 24;
		if (carry_out && chunk == 0) *(uint32_t *)carry_out = e0 | (e1 << 8) | (e2 << 16) | (e3 << 24);
	} else {
		ws = s.ws[wave];
	}
	const long long c = min(chunk, s.nw * 64 - 1);
	uint32_t st = ((const uint8_t *)(s.r + 4 * c))[ws & 255u];
	st |= (uint32_t)((const uint8_t *)(s.g + 2 * c))[(ws >> 8) & 255u] << 8;
	st |= (uint32_t)((const uint8_t *)(s.b + 4 * c))[(ws >> 16) & 255u] << 16;
	if constexpr (ALPHA == ALPHA_4) st |= (uint32_t)((const uint8_t *)(s.a + 8 * c))[ws >> 24] << 24;
	if constexpr (ALPHA == ALPHA_MOD) st |= (((ws >> 24) + s.a[c]) % 255u) << 24;
	__syncthreads();
	emit_chunk<ALPHA>(tex + (int)threadIdx.x * (L + 1), L, st, plain);
	__syncthreads();
	store_texels(tex, cnt, lsh, out + p0);
}

// The whole dither of up to SIMPLE_ONE texels in one workgroup of at most 16
// waves.
template <int COMPS, int ALPHA>
__global__ __launch_bounds__(1024) void k_simple_one(const uint8_t *__restrict__ src, int n, int plain,
                                                     const uint8_t *__restrict__ carry_in,
                                                     uint8_t *__restrict__ carry_out, uint32_t *__restrict__ out)
{
	constexpr int L = 1 << SIMPLE_ONE_LSH;
	uint32_t *tab = simple_lds, *tex = simple_lds + table_words<ALPHA>();
	__shared__ uint32_t wr[16 * 4], wg[16 * 2], wb[16 * 4], wa[16 * 8];
	const int lane = (int)(threadIdx.x & 63), wave = (int)(threadIdx.x >> 6), nw = (int)(blockDim.x >> 6);
	for (int i = (int)threadIdx.x; i < table_words<ALPHA>(); i += (int)blockDim.x) tab[i] = c_entries.t[i];
	load_texels<COMPS>(src, n, (int)blockDim.x * L, SIMPLE_ONE_LSH, tex);
	__syncthreads();
	uint32_t *mine = tex + (int)threadIdx.x * (L + 1);
	Maps<ALPHA> m;
	chunk_maps<ALPHA>(mine, min(L, max(0, n - (int)threadIdx.x * L)), tab, m);
	wave_scan(m.r);
	wave_scan(m.g);
	wave_scan(m.b);
	wave_scan(m.a);
	if (lane == 63) {
		store_map(wr, wave, m.r);
		store_map(wg, wave, m.g);
		store_map(wb, wave, m.b);
		store_map(wa, wave, m.a);
	}
	__syncthreads();
	uint32_t init = start_states(ALPHA), e0, e1, e2, e3;
	if (carry_in) init = *(const uint32_t *)carry_in;
	const uint32_t sr = scan_here<SimpleMap<3>>(wr, nw, wave, init & 255u, lane, e0);
	const uint32_t sg = scan_here<SimpleMap<2>>(wg, nw, wave, (init >> 8) & 255u, lane, e1);
	const uint32_t sb = scan_here<SimpleMap<3>>(wb, nw, wave, (init >> 16) & 255u, lane, e2);
	const uint32_t sa = scan_here<typename AlphaMap<ALPHA>::T>(wa, nw, wave, init >> 24, lane, e3);
	if (carry_out && threadIdx.x == 0) *(uint32_t *)carry_out = e0 | (e1 << 8) | (e2 << 16) | (e3 << 24);
	const uint32_t st = exclusive(m.r).at(sr) | (exclusive(m.g).at(sg) << 8) | (exclusive(m.b).at(sb) << 16) |
	                    (exclusive(m.a).at(sa) << 24);
	emit_chunk<ALPHA>(mine, L, st, plain);
	__syncthreads();
	store_texels(tex, n, SIMPLE_ONE_LSH, out);
}

// DITHER_NONE (:1269-1306)
__global__ __launch_bounds__(256) void k_quantize_none(const uint8_t *__restrict__ src, int srccomps, long long n,
                                                       int alphabits, uint32_t *__restrict__ out)
{
	const long long p = (long long)blockIdx.x * 256 + threadIdx.x;
	if (p >= n) return;
	uint32_t r, g, b, a;
	if (srccomps == 4) {
		const uint32_t t = ((const uint32_t *)src)[p];
		r = t & 255u;
		g = (t >> 8) & 255u;
		b = (t >> 16) & 255u;
		a = (t >> 24) >> (8 - alphabits);
	} else {
		const uint8_t *t = src + p * 3;
		r = t[0];
		g = t[1];
		b = t[2];
		a = (1u << alphabits) - 1u;
	}
	out[p] = (r >> 3) | ((g >> 2) << 8) | ((b >> 3) << 16) | (a << 24);
}

// ---- host launchers ----

// Texels per chunk (a power of two, as its logarithm): as few as keep the
// waves of a small image at 64, which k_simple_emit scans by itself (shorter
// chains, more lanes), else 32.
static int simple_lsh(long long n)
{
	for (int l = 3; l < 5; ++l)
		if (n <= (64LL * 64) << l) return l;
	return 5;
}

static long long simple_waves(long long n)
{
	const long long per = 64LL << simple_lsh(n);
	return (n + per - 1) / per;
}

// map registers per chunk and per wave (r, g, b and the widest alpha), and the wave states
static size_t simple_scratch_bytes(long long n)
{
	const long long nw = simple_waves(n > 0 ? n : 1);
	return (size_t)(nw * 65 * (4 + 2 + 4 + 8) + nw) * 4 + 256;
}

size_t rgb565_scratch_bytes(int w, int h, int dither, size_t fs_slab)
{
	if (dither == DITHER_FLOYDSTEINBERG) return rgb565_fs_scratch_bytes(w, h, fs_slab);
	return simple_scratch_bytes((long long)w * h);
}

template <int COMPS, int ALPHA>
static int run_simple(const uint8_t *src, long long n, int plain, void *scr, const uint8_t *carry_in,
                      uint8_t *carry_out, uint32_t *out, hipStream_t st, bool host_src)
{
	const size_t tab = (size_t)table_words<ALPHA>() * 4;
	if (n <= SIMPLE_ONE) {
		const int waves = (int)((n + (64 << SIMPLE_ONE_LSH) - 1) / (64 << SIMPLE_ONE_LSH));
		const size_t lds = tab + (size_t)waves * 64 * ((1 << SIMPLE_ONE_LSH) + 1) * 4;
		k_simple_one<COMPS, ALPHA><<<1, waves * 64, lds, st>>>(src, (int)n, plain, carry_in, carry_out, out);
		return hip_check(hipGetLastError(), "dither SIMPLE kernel");
	}
	SimpleScratch s;
	s.nw = simple_waves(n);
	uint32_t *p = (uint32_t *)scr;
	const auto take = [&](long long words) {
		uint32_t *q = p;
		p += words;
		return q;
	};
	// 16-byte aligned regions first
	s.r = take(s.nw * 64 * 4);
	s.b = take(s.nw * 64 * 4);
	s.a = take(s.nw * 64 * 8);
	s.wr = take(s.nw * 4);
	s.wb = take(s.nw * 4);
	s.wa = take(s.nw * 8);
	s.g = take(s.nw * 64 * 2);
	s.wg = take(s.nw * 2);
	s.ws = take(s.nw);
	const int lsh = simple_lsh(n), scan = s.nw <= 64;
	const unsigned grid = (unsigned)((s.nw + SIMPLE_WG / 64 - 1) / (SIMPLE_WG / 64));
	const size_t lds = (size_t)SIMPLE_WG * ((1 << lsh) + 1) * 4;
	// a source in host memory crosses the bus once: the first kernel leaves its
	// texels where the last one writes the quantized ones (256 x 256 calls 41 ->
	// 36 us; in device memory reading them twice costs less than the writes)
	k_simple_maps<COMPS, ALPHA><<<grid, SIMPLE_WG, tab + lds, st>>>(src, n, lsh, s, host_src ? out : nullptr);
	if (!scan)
		k_simple_states<ALPHA><<<ALPHA == ALPHA_PLAIN ? 3 : 4, 1024, 0, st>>>(s, carry_in, carry_out);
	if (host_src)
		k_simple_emit<4, ALPHA><<<grid, SIMPLE_WG, lds, st>>>((const uint8_t *)out, n, lsh, plain, s, scan, carry_in,
		                                                      carry_out, out);
	else
		k_simple_emit<COMPS, ALPHA><<<grid, SIMPLE_WG, lds, st>>>(src, n, lsh, plain, s, scan, carry_in, carry_out, out);
	return hip_check(hipGetLastError(), "dither SIMPLE kernels");
}

// rgb565_image with the reference's argument normalisation: srccomps other
// than 3 means 4 (:1455-1463), alphabits other than 1 and 4 means 8
// (:1437-1449), dither other than NONE and FLOYDSTEINBERG means SIMPLE
// (:1419-1431).
int launch_rgb565(const void *d_src, int srccomps, int w, int h, int alphabits, int dither, void *d_out,
                  void *d_scratch, hipStream_t st, const void *d_carry_in, void *d_carry_out, bool host_src,
                  const FsRun &fs)
{
	if (srccomps != 3) srccomps = 4;
	if (alphabits != 1 && alphabits != 4) alphabits = 8;
	if (dither != DITHER_NONE && dither != DITHER_FLOYDSTEINBERG) dither = DITHER_SIMPLE;
	const long long n = (long long)w * h;
	if (n <= 0) return 0;
	const uint8_t *src = (const uint8_t *)d_src;
	uint32_t *out = (uint32_t *)d_out;
	if (dither == DITHER_NONE) {
		k_quantize_none<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(src, srccomps, n, alphabits, out);
		return hip_check(hipGetLastError(), "quantize kernel");
	}
	if (dither == DITHER_FLOYDSTEINBERG) {
		if (d_carry_in || d_carry_out)
			return set_error(S2TC_E_ARG, "the Floyd-Steinberg dither does not run in bands");
		return launch_rgb565_fs(src, srccomps, w, h, alphabits, (uint8_t *)d_out, d_scratch, st, fs);
	}
	const uint8_t *ci = (const uint8_t *)d_carry_in;
	uint8_t *co = (uint8_t *)d_carry_out;
	if (srccomps == 3) return run_simple<3, ALPHA_PLAIN>(src, n, (1 << alphabits) - 1, d_scratch, ci, co, out, st, host_src);
	if (alphabits == 1) return run_simple<4, ALPHA_MOD>(src, n, 0, d_scratch, ci, co, out, st, host_src);
	if (alphabits == 4) return run_simple<4, ALPHA_4>(src, n, 0, d_scratch, ci, co, out, st, host_src);
	return run_simple<4, ALPHA_PLAIN>(src, n, -1, d_scratch, ci, co, out, st, host_src);
}

}  // namespace s2tc
