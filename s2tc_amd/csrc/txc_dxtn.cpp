// txc_dxtn.cpp - the reference-compatible C ABI (txc_dxtn.h, s2tc_algorithm.h).
//
// tx_compress_dxtn follows s2tc_libtxc_dxtn.cpp:142-299: environment
// configuration read on every call, GL format switch, rgb565_image, the
// raster block loop and the destination row padding rule.  The quantization
// and the block loop run on the GPU; the host copies the source into pinned
// memory and lays out the destination rows from the blocks.  Each call borrows a
// context (stream + device buffers) from a pool, so concurrent callers on
// different threads do not share buffers.
#include "s2tc_internal.h"

#include <algorithm>
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <strings.h>
#include <thread>
#include <vector>

#include "s2tc_algorithm.h"
#include "staging.h"
#include "txc_dxtn.h"

namespace s2tc {

struct DevBuf {
	void *p = nullptr;
	size_t cap = 0;
	int ensure(size_t n)
	{
		if (n <= cap) return 0;
		if (p) (void)hipFree(p);
		p = nullptr;
		cap = 0;
		n = (n + 4095) & ~(size_t)4095;
		if (int r = hip_check(hipMalloc(&p, n), "hipMalloc")) return r;
		cap = n;
		return 0;
	}
	void release()
	{
		if (p) (void)hipFree(p);
		p = nullptr;
		cap = 0;
	}
};

// Pinned host memory (hipHostMalloc): staging for the host-buffer entry
// points that copies and kernels (at `dev`) reach, grown on demand and kept
// with the context.
struct HostBuf {
	void *p = nullptr, *dev = nullptr;
	size_t cap = 0;
	int ensure(size_t n)
	{
		if (n <= cap) return 0;
		if (p) (void)hipHostFree(p);
		p = nullptr;
		cap = 0;
		n = (n + 4095) & ~(size_t)4095;
		if (int r = hip_check(hipHostMalloc(&p, n, hipHostMallocMapped), "hipHostMalloc")) return r;
		if (int r = hip_check(hipHostGetDevicePointer(&dev, p, 0), "hipHostGetDevicePointer")) {
			(void)hipHostFree(p);
			p = nullptr;
			return r;
		}
		cap = n;
		return 0;
	}
	uint8_t *data() const { return (uint8_t *)p; }
};

// How a call's host data reaches the kernels and comes back, by size; measured
// (MI355X, whole calls, against a copy into staging, a DMA, the kernels, a DMA
// back and the rows laid out, one after the other):
//   up to kDirectMax, the kernels read the pinned copy of the source, and write
//   blocks of up to kDirectMax to pinned memory: 256 x 256 RGBA quick 36 -> 21
//   us, with the SIMPLE dither 50 -> 36 us (at 1 MiB the Floyd-Steinberg dither
//   loses: 189 -> 266 us for its short reads, the others change little);
//   up to kBandMin, the upload kernel runs over each half while the other is
//   copied: 1024 x 1024 SIMPLE 216 -> 175 us (four pieces: the same);
//   above, in bands (encode_host_bands) with uploads of kChunk through a ring of
//   kRing pinned buffers: 2048 x 2048 NONE 601 -> 483 us, 4096 x 4096 DXT5
//   SIMPLE 2.04 -> 1.86 ms (2 MiB: 1.93 ms; 512 KiB: 1.99 ms).  In bands from 4
//   MiB on, 1024 x 1024 SIMPLE took 253 us: starting the threads and the
//   smaller launches cost more than the overlap gives.
static const size_t kDirectMax = 512u << 10;
static const size_t kBandMin = 8u << 20;
static const size_t kChunk = 1u << 20, kRing = 12;
// Host threads (the caller's included) that copy; three to six measure alike,
// eight are 5% slower.
static const unsigned kCopyThreads = 4;
// Bands whose blocks may be on their way back.
static const int kOutRing = 4;

static unsigned copy_helpers()
{
	const unsigned hw = std::thread::hardware_concurrency();
	return std::max(1u, std::min(kCopyThreads, hw ? hw : 1u)) - 1;
}

struct Ctx {
	hipStream_t stream = nullptr;
	hipStream_t copy_stream[2] = {};    // uploads of a call encoded in bands (created on first use)
	DevBuf src, q, out, scratch;
	HostBuf in_stage, host_out;
	hipEvent_t stage_ev[kRing] = {};    // last upload out of each buffer of in_stage
	hipEvent_t out_ev[kOutRing] = {};   // encoded bands
	// one mapped pinned page: per-block calls, whose kernel reads the block's
	// texels from it (offset 0) and writes its encoding to it (offset 64), and the
	// word of FsRun (kPageGaveUp)
	uint8_t *page = nullptr;
	uint8_t *page_dev = nullptr;
	int ensure_page()
	{
		if (page) return 0;
		if (int r = hip_check(hipHostMalloc((void **)&page, 4096, hipHostMallocMapped), "hipHostMalloc")) return r;
		const int r = hip_check(hipHostGetDevicePointer((void **)&page_dev, page, 0), "hipHostGetDevicePointer");
		if (r) {
			(void)hipHostFree(page);
			page = nullptr;
		}
		return r;
	}
};
static const size_t kPageGaveUp = 128;

// Looks that a wait of the Floyd-Steinberg dither lasts at most (test hook).
static thread_local unsigned t_fs_polls = FS_POLLS;

// The waits of a call's dither: before its launch, and after its synchronize.
static int fs_begin(Ctx *c, int dither, FsRun &run)
{
	if (dither != DITHER_FLOYDSTEINBERG) return 0;
	if (int r = c->ensure_page()) return r;
	*(volatile uint32_t *)(c->page + kPageGaveUp) = 0;
	run.gave_up = (uint32_t *)(c->page_dev + kPageGaveUp);
	run.polls = t_fs_polls;
	return 0;
}
static int fs_end(Ctx *c, int dither)
{
	if (dither != DITHER_FLOYDSTEINBERG || !*(volatile uint32_t *)(c->page + kPageGaveUp)) return 0;
	return set_error(S2TC_E_HIP, "the Floyd-Steinberg dither's waves waited too long for each other");
}

// Whether the work that an event follows is done (a query that is not leaves no
// error behind for the next launch to find).
static bool event_done(hipEvent_t ev)
{
	if (hipEventQuery(ev) == hipSuccess) return true;
	(void)hipGetLastError();
	return false;
}

// Upload of a source in chunks through the ring of pinned buffers: while the
// upload kernel of a chunk runs, the host threads copy the next ones (one host
// thread alone copies pageable memory well below the link rate).  A buffer is
// refilled only after the event of the upload that last read it; a call leaves
// none behind, so the buffers start out free.  Chunks alternate between st0 and
// st1: two streams hide the gap between one stream's kernels.  on_chunk (if
// given) learns of every queued chunk and how many leading bytes are then on
// their way, after the next chunk is queued.
static int upload_chunks(Ctx *c, CopyCrew &crew, void *dst, hipStream_t st0, hipStream_t st1,
                         const std::function<int(size_t, size_t)> &on_chunk = nullptr)
{
	for (auto &ev : c->stage_ev)
		if (!ev)
			if (int r = hip_check(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "hipEventCreate")) return r;
	size_t open = std::min(crew.nchunks, crew.ring);
	crew.open_chunks(open);
	for (size_t i = 0; i < crew.nchunks; ++i) {
		while (!crew.chunk_copied(i))
			if (!crew.step()) std::this_thread::yield();
		const size_t off = i * crew.chunk, len = crew.chunk_len(i);
		const hipStream_t st = i & 1 ? st1 : st0;
		if (int r = launch_pull((uint8_t *)dst + off, (uint8_t *)c->in_stage.dev + crew.ring_offset(i), len, st))
			return r;
		if (on_chunk || crew.nchunks > crew.ring)
			if (int r = hip_check(hipEventRecord(c->stage_ev[i % crew.ring], st), "hipEventRecord")) return r;
		// what the previous chunk completed, while this one is on its way
		if (on_chunk && i)
			if (int r = on_chunk(i - 1, off)) return r;
		// open the buffers whose upload ended; the next chunk's by waiting
		while (open < crew.nchunks && open <= i + crew.ring) {
			hipEvent_t ev = c->stage_ev[open % crew.ring];
			if (open == i + 1) {
				if (int r = hip_check(hipEventSynchronize(ev), "hipEventSynchronize")) return r;
			} else if (!event_done(ev)) {
				break;
			}
			crew.open_chunks(++open);
		}
	}
	return on_chunk ? on_chunk(crew.nchunks - 1, crew.n) : 0;
}

// host -> device upload of a caller's buffer on the context's stream
static int upload(Ctx *c, void *dst, const void *src, size_t n)
{
	if (n <= 2 * kDirectMax) {
		if (int r = c->in_stage.ensure(n)) return r;
		memcpy(c->in_stage.p, src, n);
		return launch_pull(dst, c->in_stage.dev, n, c->stream);
	}
	// halves, or pieces of 4 MiB by several threads
	const size_t chunk = std::min(((n + 1) / 2 + 4095) & ~(size_t)4095, (size_t)4 << 20);
	const size_t ring = std::min((size_t)4, (n + chunk - 1) / chunk);
	if (int r = c->in_stage.ensure(ring * chunk)) return r;
	CopyCrew crew((const uint8_t *)src, n, c->in_stage.data(), chunk, ring);
	if (n > 2 * chunk) crew.start(copy_helpers());
	return upload_chunks(c, crew, dst, c->stream, c->stream);
}

static std::mutex g_pool_mu;
static std::vector<Ctx *> g_pool;

static Ctx *ctx_acquire()
{
	{
		std::lock_guard<std::mutex> lk(g_pool_mu);
		if (!g_pool.empty()) {
			Ctx *c = g_pool.back();
			g_pool.pop_back();
			return c;
		}
	}
	Ctx *c = new Ctx;
	if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
		delete c;
		return nullptr;
	}
	return c;
}

// Scratch that an idle context keeps: that of 4096 x 4096 with the
// Floyd-Steinberg dither (134 MiB); to give back and to allocate more takes 0.27
// ms, in calls of 5 ms and more.
static const size_t kKeepScratch = (size_t)192 << 20;

static void ctx_release(Ctx *c)
{
	if (c->scratch.cap > kKeepScratch) c->scratch.release();
	std::lock_guard<std::mutex> lk(g_pool_mu);
	g_pool.push_back(c);
}

struct CtxGuard {
	Ctx *c;
	CtxGuard() : c(ctx_acquire()) {}
	~CtxGuard()
	{
		if (c) ctx_release(c);
	}
};

// Scratch of a dither.  That of the Floyd-Steinberg dither is FsRun::slab and
// somewhat more: where the device has not that much left, what idle contexts keep
// is given back, and then the slabs get smaller, to one band of rows if need be.
static thread_local size_t t_fs_scratch_max = ~(size_t)0;  // test hook

static int dither_scratch(Ctx *c, int w, int h, int dither, FsRun &run)
{
	size_t n = rgb565_scratch_bytes(w, h, dither, run.slab);
	if (dither != DITHER_FLOYDSTEINBERG) return c->scratch.ensure(n);
	for (bool trimmed = false;;) {
		const int r = n > t_fs_scratch_max ? set_error(S2TC_E_HIP, "no scratch of %zu bytes", n) : c->scratch.ensure(n);
		if (!r) return 0;
		(void)hipGetLastError();  // not for the next launch to find
		if (!trimmed) {
			std::lock_guard<std::mutex> lk(g_pool_mu);
			for (Ctx *idle : g_pool) idle->scratch.release();
			trimmed = true;
			continue;
		}
		const size_t before = n;
		while (n == before) {
			if (!run.slab) return r;
			run.slab /= 4;
			n = rgb565_scratch_bytes(w, h, dither, run.slab);
		}
	}
}

// Environment configuration of s2tc_libtxc_dxtn.cpp:156-216.
struct EnvConfig {
	int cd = CD_WAVG, nrandom = -1, refine = REFINE_ALWAYS, dither = DITHER_SIMPLE;
	uint64_t seed = 0;
};

static EnvConfig read_env()
{
	EnvConfig e;
	if (const char *v = getenv("S2TC_DITHER_MODE")) {
		if (!strcasecmp(v, "NONE")) e.dither = DITHER_NONE;
		else if (!strcasecmp(v, "SIMPLE")) e.dither = DITHER_SIMPLE;
		else if (!strcasecmp(v, "FLOYDSTEINBERG")) e.dither = DITHER_FLOYDSTEINBERG;
		else fprintf(stderr, "Invalid dither mode: %s\n", v);
	}
	if (const char *v = getenv("S2TC_COLORDIST_MODE")) {
		static const char *names[] = {"RGB", "YUV", "SRGB", "SRGB_MIXED", "AVG", "WAVG", "W0AVG", "NORMALMAP"};
		int found = -1;
		for (int i = 0; i < 8; ++i)
			if (!strcasecmp(v, names[i])) found = i;
		if (found >= 0) e.cd = found;
		else fprintf(stderr, "Invalid color dist mode: %s\n", v);
	}
	if (const char *v = getenv("S2TC_RANDOM_COLORS")) e.nrandom = atoi(v);
	if (const char *v = getenv("S2TC_REFINE_COLORS")) {
		if (!strcasecmp(v, "NEVER")) e.refine = REFINE_NEVER;
		else if (!strcasecmp(v, "ALWAYS")) e.refine = REFINE_ALWAYS;
		else if (!strcasecmp(v, "LOOP")) e.refine = REFINE_LOOP;
		else fprintf(stderr, "Invalid refinement mode: %s\n", v);
	}
	if (const char *v = getenv("S2TC_RANDOM_SEED")) e.seed = strtoull(v, nullptr, 0);
	return e;
}

// Rows per band of a large call (a multiple of 4: whole block rows): the
// upload of later rows overlaps the dither and encode of earlier ones.  At
// least 512 rows, and at least 2^18 blocks per band, which the one-lane-per-
// block encoders need to fill the GPU (8192 x 4096 with 2^17: 2.6 instead of
// 2.4 ms), or half the image.
static int band_rows(int width, int height)
{
	const long long r = std::max(512LL, ((1LL << 22) + width - 1) / width);
	return (int)((std::min(r, (height + 1LL) / 2) + 3) & ~3LL);
}

// Large sources (above kBandMin) with the NONE or SIMPLE dither: the uploads
// run on the copy streams, and each band of rows is quantized and encoded on the
// compute stream as soon as its rows are uploaded, beside the later uploads (a
// band computes in less time than it uploads).  SIMPLE carries its error state
// from band to band on the device; the encoder numbers the blocks of a band from
// the band's first block, so the random candidates are those of the whole image,
// and writes them to pinned memory itself.  No stream for each kind of work: the
// hardware queues of a process are few, and streams that share one wait for each
// other.  The rows of finished bands go to rows_dest (if given) while later ones
// are on their way.
static int encode_host_bands(Ctx *c, int srccomps, int width, int height, const uint8_t *src, int dxt,
                             const EncodeArgs &base, int dither, int alphabits, uint8_t *rows_dest, size_t row_pitch)
{
	const int brows = band_rows(width, height);
	const size_t row_bytes = (size_t)width * srccomps;
	const size_t n = (size_t)width * height;
	const int bw = (width + 3) / 4, bb = block_bytes(dxt);
	// the last rows in bands of half the size: what is left to do after the last
	// upload is short
	const int full = (height - 1) / brows * brows, half = std::max(4, brows / 2 & ~3);
	const int nbands = full / brows + (height - full + half - 1) / half;
	const auto band_row = [&](int b) {
		return (long long)b * brows <= full ? b * brows
		                                    : (int)std::min((long long)height, full + (b - full / brows) * (long long)half);
	};
	const bool fused = dither == DITHER_NONE && srccomps == 4;
	size_t scratch = 0;
	for (int b = 0; b < nbands; ++b)
		scratch = std::max(scratch, rgb565_scratch_bytes(width, band_row(b + 1) - band_row(b), dither));
	if (!fused) {
		if (int r = c->q.ensure(n * 4)) return r;
		if (int r = c->scratch.ensure(scratch + 256)) return r;
	}
	for (auto &st : c->copy_stream)
		if (!st)
			if (int r = hip_check(hipStreamCreateWithFlags(&st, hipStreamNonBlocking), "hipStreamCreate")) return r;
	for (auto &ev : c->out_ev)
		if (!ev)
			if (int r = hip_check(hipEventCreateWithFlags(&ev, hipEventDisableTiming), "hipEventCreate")) return r;
	if (int r = c->in_stage.ensure(kRing * kChunk)) return r;
	CopyCrew crew(src, n * srccomps, c->in_stage.data(), kChunk, kRing);
	if (rows_dest) crew.set_rows(rows_dest, c->host_out.data(), (size_t)bw * bb, row_pitch, (height + 3) / 4);
	crew.start(copy_helpers());
	uint8_t *carry = (uint8_t *)c->scratch.p + scratch;
	int next = 0, back = 0;  // bands launched, bands whose blocks have come back
	// opens the rows of the bands that came back; waits for those before `until`
	auto collect = [&](int until) -> int {
		while (back < next) {
			hipEvent_t ev = c->out_ev[back % kOutRing];
			if (back < until) {
				if (int r = hip_check(hipEventSynchronize(ev), "hipEventSynchronize")) return r;
			} else if (!event_done(ev)) {
				break;
			}
			++back;
			crew.open_rows((band_row(back) + 3) / 4);
		}
		return 0;
	};
	auto on_chunk = [&](size_t chunk, size_t uploaded) -> int {
		bool waited = false;
		if (int r = collect(0)) return r;
		while (next < nbands && (size_t)band_row(next + 1) * row_bytes <= uploaded) {
			if (!waited) {
				// the last chunk of either copy stream
				for (size_t i = chunk ? chunk - 1 : 0; i <= chunk; ++i)
					if (int r = hip_check(hipStreamWaitEvent(c->stream, c->stage_ev[i % crew.ring], 0),
					                      "hipStreamWaitEvent"))
						return r;
				waited = true;
			}
			const int r0 = band_row(next), rows = band_row(next + 1) - r0;
			const uint8_t *bsrc = (const uint8_t *)c->src.p + (size_t)r0 * row_bytes;
			EncodeArgs a = base;
			a.height = rows;
			a.block_index_base = (uint32_t)((size_t)(r0 / 4) * bw);
			if (fused) {
				a.src = bsrc;
				a.src_kind = S2TC_SRC_RGBA8;
			} else {
				uint8_t *bq = (uint8_t *)c->q.p + (size_t)r0 * width * 4;
				if (int r = launch_rgb565(bsrc, srccomps, width, rows, alphabits, dither, bq, c->scratch.p, c->stream,
				                          next > 0 ? carry + 4 * (next & 1) : nullptr, carry + 4 * ((next + 1) & 1)))
					return r;
				a.src = bq;
				a.src_kind = S2TC_SRC_QUANTIZED;
			}
			a.dst = (uint8_t *)c->host_out.dev + (size_t)(r0 / 4) * bw * bb;
			if (int r = launch_encode(a, c->stream)) return r;
			if (int r = collect(next + 1 - kOutRing)) return r;
			if (int r = hip_check(hipEventRecord(c->out_ev[next % kOutRing], c->stream), "hipEventRecord")) return r;
			++next;
		}
		return 0;
	};
	if (int r = upload_chunks(c, crew, c->src.p, c->copy_stream[0], c->copy_stream[1], on_chunk)) return r;
	if (next != nbands) return set_error(S2TC_E_ARG, "banded encode: %d of %d bands launched", next, nbands);
	while (back < nbands)
		if (int r = collect(back + 1)) return r;
	while (rows_dest && !crew.rows_copied())
		if (!crew.step()) std::this_thread::yield();
	return 0;
}

static int encode_host_image_on(Ctx *c, int srccomps, int width, int height, const uint8_t *src, int dxt, int cd,
                                int nrandom, int refine, int dither, uint64_t seed, uint8_t *rows_dest,
                                size_t row_pitch, bool &rows_written);

// Whole-image encode of host data on the context's stream; writes the
// blocks in raster order to c->host_out, and their rows to rows_dest (if given)
// where it says so in rows_written.  On an error every stream of the
// context is drained before the context goes back to the pool, so that no
// launch of this call still uses its buffers when the next call resizes them.
static int encode_host_image(Ctx *c, int srccomps, int width, int height, const uint8_t *src, int dxt, int cd,
                             int nrandom, int refine, int dither, uint64_t seed, uint8_t *rows_dest, size_t row_pitch,
                             bool &rows_written)
{
	const int rc = encode_host_image_on(c, srccomps, width, height, src, dxt, cd, nrandom, refine, dither, seed,
	                                    rows_dest, row_pitch, rows_written);
	if (rc) {
		for (hipStream_t st : {c->stream, c->copy_stream[0], c->copy_stream[1]})
			if (st) (void)hipStreamSynchronize(st);
	}
	return rc;
}

static int encode_host_image_on(Ctx *c, int srccomps, int width, int height, const uint8_t *src, int dxt, int cd,
                                int nrandom, int refine, int dither, uint64_t seed, uint8_t *rows_dest,
                                size_t row_pitch, bool &rows_written)
{
	rows_written = false;
	if (srccomps != 3) srccomps = 4;
	if (dither != DITHER_NONE && dither != DITHER_FLOYDSTEINBERG) dither = DITHER_SIMPLE;
	const size_t n = (size_t)width * height;
	const size_t nb = (size_t)((width + 3) / 4) * ((height + 3) / 4);
	const size_t obytes = nb * block_bytes(dxt);
	const int alphabits = dxt == DXT1 ? 1 : dxt == DXT3 ? 4 : 8;
	const bool bands = dither != DITHER_FLOYDSTEINBERG && height > 8 && n * srccomps > kBandMin;
	const bool direct = n * srccomps <= kDirectMax, direct_out = bands || obytes <= kDirectMax;
	if (int r = direct ? c->in_stage.ensure(n * srccomps) : c->src.ensure(n * srccomps)) return r;
	const void *d_src = direct ? c->in_stage.dev : c->src.p;
	if (int r = c->host_out.ensure(obytes)) return r;
	if (int r = direct_out ? 0 : c->out.ensure(obytes)) return r;
	EncodeArgs a{};
	a.dst = direct_out ? c->host_out.dev : c->out.p;
	a.width = width;
	a.height = height;
	a.dxt = dxt;
	a.cd = cd;
	a.nrandom = nrandom;
	a.refine = refine;
	a.seed = seed;
	if (bands) {
		// the blocks are in c->host_out once the last band is encoded
		if (int r = encode_host_bands(c, srccomps, width, height, src, dxt, a, dither, alphabits, rows_dest, row_pitch))
			return r;
		rows_written = rows_dest != nullptr;
		return 0;
	}
	if (direct) memcpy(c->in_stage.p, src, n * srccomps);
	else if (int r = upload(c, c->src.p, src, n * srccomps)) return r;
	if (dither == DITHER_NONE && srccomps == 4) {
		a.src = d_src;  // quantization fused into the encoder's loads
		a.src_kind = S2TC_SRC_RGBA8;
	} else {
		if (int r = c->q.ensure(n * 4)) return r;
		FsRun run;
		if (int r = fs_begin(c, dither, run)) return r;
		if (int r = dither_scratch(c, width, height, dither, run)) return r;
		if (int r = launch_rgb565(d_src, srccomps, width, height, alphabits, dither, c->q.p, c->scratch.p, c->stream,
		                          nullptr, nullptr, direct, run))
			return r;
		a.src = c->q.p;
		a.src_kind = S2TC_SRC_QUANTIZED;
	}
	if (int r = launch_encode(a, c->stream)) return r;
	if (!direct_out)
		if (int r = hip_check(hipMemcpyAsync(c->host_out.data(), c->out.p, obytes, hipMemcpyDeviceToHost, c->stream),
		                      "D2H"))
			return r;
	if (int r = hip_check(hipStreamSynchronize(c->stream), "hipStreamSynchronize")) return r;
	return fs_end(c, dither);
}

// ---- per-block entry points of s2tc_encode_block_func ----

static thread_local uint32_t t_block_index = 0;

static void encode_one_block(unsigned char *out, const unsigned char *rgba, int iw, int w, int h, int nrandom,
                             int dxt, int cd, int fast, int refine)
{
	CtxGuard g;
	Ctx *c = g.c;
	const uint32_t bidx = t_block_index++;
	if (!c) {
		fprintf(stderr, "s2tc: cannot create a HIP stream\n");
		return;
	}
	if (w < 1 || h < 1 || w > 4 || h > 4) return;
	const int bs = block_bytes(dxt);
	int r = c->ensure_page();
	if (!r) {
		// the block's rows, packed, where the kernel reads them over the bus
		for (int y = 0; y < h; ++y) memcpy(c->page + y * w * 4, rgba + (size_t)y * iw * 4, (size_t)w * 4);
		// A one-block image whose only block has index bidx in the generator.
		// The selection-time mode is kept: quick mode runs with nrandom < 0,
		// MODE_NORMAL with max(nrandom, 0) extra candidates.
		uint8_t *dev = c->page_dev;
		EncodeArgs a{dev, dev + 64, S2TC_SRC_QUANTIZED, w, h, dxt, cd, fast ? -1 : (nrandom > 0 ? nrandom : 0),
		             refine, 0, 0};
		const char *sv = getenv("S2TC_RANDOM_SEED");
		a.seed = sv ? strtoull(sv, nullptr, 0) : 0;
		a.block_index_base = bidx;
		r = launch_encode(a, c->stream);
	}
	if (!r) r = hip_check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
	if (r) {
		fprintf(stderr, "s2tc: %s\n", s2tc_amd_last_error());
		return;
	}
	memcpy(out, c->page + 64, bs);
}

template <int DXT, int CD, int FAST, int REFINE>
static void block_fn(unsigned char *out, const unsigned char *rgba, int iw, int w, int h, int nrandom)
{
	encode_one_block(out, rgba, iw, w, h, nrandom, DXT, CD, FAST, REFINE);
}

template <int DXT, int CD, int FAST>
static s2tc_encode_block_func_t pick_refine(int refine)
{
	switch (refine) {
	case REFINE_NEVER: return block_fn<DXT, CD, FAST, REFINE_NEVER>;
	case REFINE_LOOP: return block_fn<DXT, CD, FAST, REFINE_LOOP>;
	default: return block_fn<DXT, CD, FAST, REFINE_ALWAYS>;
	}
}

template <int DXT, int CD>
static s2tc_encode_block_func_t pick_mode(int nrandom, int refine)
{
	if (CD == CD_NORMALMAP || nrandom >= 0) return pick_refine<DXT, CD, 0>(refine);
	return pick_refine<DXT, CD, CD == CD_NORMALMAP ? 0 : 1>(refine);
}

template <int CD>
static s2tc_encode_block_func_t pick_dxt(int dxt, int nrandom, int refine)
{
	switch (dxt) {
	case DXT1: return pick_mode<DXT1, CD>(nrandom, refine);
	case DXT3: return pick_mode<DXT3, CD>(nrandom, refine);
	default: return pick_mode<DXT5, CD>(nrandom, refine);
	}
}

}  // namespace s2tc

using namespace s2tc;

extern "C" {

void tx_compress_dxtn(GLint srccomps, GLint width, GLint height, const GLubyte *srcPixData, GLenum destformat,
                      GLubyte *dest, GLint dstRowStride)
{
	const EnvConfig e = read_env();
	int dxt, k;
	switch (destformat) {
	case 0x83F0: /* GL_COMPRESSED_RGB_S3TC_DXT1_EXT */
	case 0x83F1: /* GL_COMPRESSED_RGBA_S3TC_DXT1_EXT */
		dxt = s2tc::DXT1;
		k = 2;
		break;
	case 0x83F2: dxt = s2tc::DXT3; k = 4; break;
	case 0x83F3: dxt = s2tc::DXT5; k = 4; break;
	default:
		fprintf(stderr, "libdxtn: Bad dstFormat %d in tx_compress_dxtn\n", destformat);
		return;
	}
	if (width <= 0 || height <= 0) return;
	CtxGuard g;
	if (!g.c) {
		fprintf(stderr, "s2tc: cannot create a HIP stream\n");
		return;
	}
	// destination layout with dstRowDiff (s2tc_libtxc_dxtn.cpp:243, :261, :279)
	const int bs = block_bytes(dxt);
	const int bw = (width + 3) / 4, bh = (height + 3) / 4;
	const long rowdiff = dstRowStride >= width * k ? (long)dstRowStride - (long)((width + 3) & ~3) * k : 0;
	const size_t rowbytes = (size_t)bw * bs;
	// rows that overlap each other (a negative row gap) are written in order, and
	// rows over the source after the whole source is read
	const uintptr_t s0 = (uintptr_t)srcPixData, s1 = s0 + (size_t)width * height * (srccomps == 3 ? 3 : 4);
	const uintptr_t d0 = (uintptr_t)dest, d1 = d0 + (rowbytes + (size_t)std::max(rowdiff, 0L)) * (size_t)bh;
	const bool early = rowdiff >= 0 && (d1 <= s0 || s1 <= d0);
	bool written = false;
	if (int r = encode_host_image(g.c, srccomps, width, height, srcPixData, dxt, e.cd, e.nrandom, e.refine, e.dither,
	                              e.seed, early ? dest : nullptr, rowbytes + (size_t)rowdiff, written)) {
		fprintf(stderr, "s2tc: tx_compress_dxtn failed (%d): %s\n", r, s2tc_amd_last_error());
		return;
	}
	if (written) return;
	const uint8_t *hout = g.c->host_out.data();
	if (rowdiff < 0 || rowbytes * (size_t)bh < (2u << 20)) {
		for (int by = 0; by < bh; ++by)
			memcpy(dest + ((long)rowbytes + rowdiff) * by, hout + (size_t)by * rowbytes, rowbytes);
		return;
	}
	// disjoint rows: several host threads
	CopyCrew crew(nullptr, 0, nullptr, 1, 1);
	crew.set_rows(dest, hout, rowbytes, rowbytes + (size_t)rowdiff, bh);
	crew.open_rows(bh);
	crew.start(copy_helpers());
	while (!crew.rows_copied())
		if (!crew.step()) std::this_thread::yield();
}

void rgb565_image(unsigned char *out, const unsigned char *rgba, int w, int h, int srccomps, int alphabits,
                  enum DitherMode dither)
{
	if (w <= 0 || h <= 0) return;
	CtxGuard g;
	Ctx *c = g.c;
	if (!c) {
		fprintf(stderr, "s2tc: cannot create a HIP stream\n");
		return;
	}
	const int sc = srccomps == 3 ? 3 : 4;
	const size_t n = (size_t)w * h;
	int r = c->src.ensure(n * sc);
	if (!r) r = c->q.ensure(n * 4);
	FsRun run;
	if (!r) r = fs_begin(c, (int)dither, run);
	if (!r) r = dither_scratch(c, w, h, (int)dither, run);
	if (!r) r = upload(c, c->src.p, rgba, n * sc);
	if (!r)
		r = launch_rgb565(c->src.p, sc, w, h, alphabits, (int)dither, c->q.p, c->scratch.p, c->stream, nullptr, nullptr,
		                  false, run);
	if (!r) r = hip_check(hipMemcpyAsync(out, c->q.p, n * 4, hipMemcpyDeviceToHost, c->stream), "D2H");
	if (!r) r = hip_check(hipStreamSynchronize(c->stream), "hipStreamSynchronize");
	if (r) (void)hipStreamSynchronize(c->stream);
	else r = fs_end(c, (int)dither);
	if (r) fprintf(stderr, "s2tc: rgb565_image failed (%d): %s\n", r, s2tc_amd_last_error());
}

s2tc_encode_block_func_t s2tc_encode_block_func(enum DxtMode dxt, ColorDistMode cd, int nrandom,
                                                enum RefinementMode refine)
{
	switch ((int)cd) {
	case CD_RGB: return pick_dxt<CD_RGB>(dxt, nrandom, refine);
	case CD_YUV: return pick_dxt<CD_YUV>(dxt, nrandom, refine);
	case CD_SRGB: return pick_dxt<CD_SRGB>(dxt, nrandom, refine);
	case CD_SRGB_MIXED: return pick_dxt<CD_SRGB_MIXED>(dxt, nrandom, refine);
	case CD_AVG: return pick_dxt<CD_AVG>(dxt, nrandom, refine);
	case CD_W0AVG: return pick_dxt<CD_W0AVG>(dxt, nrandom, refine);
	case CD_NORMALMAP: return pick_dxt<CD_NORMALMAP>(dxt, nrandom, refine);
	default: return pick_dxt<CD_WAVG>(dxt, nrandom, refine);
	}
}

void s2tc_amd_set_block_index(unsigned int index) { t_block_index = index; }

void s2tc_amd_debug_set_fs_polls(unsigned polls) { t_fs_polls = std::min(polls, FS_POLLS); }

void s2tc_amd_debug_set_fs_scratch_max(size_t bytes) { t_fs_scratch_max = bytes; }

// ---- S2TC decoders (s2tc_libtxc_dxtn.cpp:35-140) ----

static inline void expand565(unsigned c, GLubyte *t)
{
	unsigned r = (c >> 11) & 0x1f, g = (c >> 5) & 0x3f, b = c & 0x1f;
	t[0] = (GLubyte)((r << 3) | (r >> 2));
	t[1] = (GLubyte)((g << 2) | (g >> 4));
	t[2] = (GLubyte)((b << 3) | (b >> 2));
}

static inline const GLubyte *block_at(GLint stride, const GLubyte *pix, GLint i, GLint j, int bs)
{
	return pix + ((size_t)((stride + 3) >> 2) * (size_t)(j >> 2) + (size_t)(i >> 2)) * bs;
}

// colour of an S2TC block: 0 -> c0, 1 -> c1, 2/3 -> checkerboard of c0/c1;
// with dxt1_black, index 3 with c1 >= c0 is black (transparent for RGBA).
static inline unsigned s2tc_color(const GLubyte *cb, GLint i, GLint j, bool dxt1, bool &black)
{
	const unsigned c0 = cb[0] | (cb[1] << 8), c1 = cb[2] | (cb[3] << 8);
	const int idx = (cb[4 + (j & 3)] >> (2 * (i & 3))) & 3;
	black = false;
	if (idx == 0) return c0;
	if (idx == 1) return c1;
	if (dxt1 && idx == 3 && c1 >= c0) {
		black = true;
		return 0;
	}
	return ((i ^ j) & 1) ? c1 : c0;
}

void fetch_2d_texel_rgb_dxt1(GLint srcRowStride, const GLubyte *pixdata, GLint i, GLint j, GLvoid *texel)
{
	GLubyte *t = (GLubyte *)texel;
	bool black;
	expand565(s2tc_color(block_at(srcRowStride, pixdata, i, j, 8), i, j, true, black), t);
	t[3] = 255;
}

void fetch_2d_texel_rgba_dxt1(GLint srcRowStride, const GLubyte *pixdata, GLint i, GLint j, GLvoid *texel)
{
	GLubyte *t = (GLubyte *)texel;
	bool black;
	expand565(s2tc_color(block_at(srcRowStride, pixdata, i, j, 8), i, j, true, black), t);
	t[3] = black ? 0 : 255;
}

void fetch_2d_texel_rgba_dxt3(GLint srcRowStride, const GLubyte *pixdata, GLint i, GLint j, GLvoid *texel)
{
	GLubyte *t = (GLubyte *)texel;
	const GLubyte *blk = block_at(srcRowStride, pixdata, i, j, 16);
	bool black;
	expand565(s2tc_color(blk + 8, i, j, false, black), t);
	const int a = (blk[(j & 3) * 2 + ((i & 3) >> 1)] >> (4 * (i & 1))) & 0x0f;
	t[3] = (GLubyte)(a | (a << 4));
}

void fetch_2d_texel_rgba_dxt5(GLint srcRowStride, const GLubyte *pixdata, GLint i, GLint j, GLvoid *texel)
{
	GLubyte *t = (GLubyte *)texel;
	const GLubyte *blk = block_at(srcRowStride, pixdata, i, j, 16);
	bool black;
	expand565(s2tc_color(blk + 8, i, j, false, black), t);
	unsigned a = blk[0];
	const unsigned a1 = blk[1];
	uint64_t bits = 0;
	for (int q = 0; q < 6; ++q) bits |= (uint64_t)blk[2 + q] << (8 * q);
	const int ab = (int)((bits >> (3 * ((j & 3) * 4 + (i & 3)))) & 7);
	// index 6 is 0 and 7 is 255 in 6-value mode (a1 >= a0); otherwise 6 falls
	// through to 7's test and both fall through to the checkerboard (:130-137)
	if (ab == 1) a = a1;
	else if (ab == 6 && a1 >= a) a = 0;
	else if ((ab == 6 || ab == 7) && a1 >= a) a = 255;
	else if (ab != 0 && ((i ^ j) & 1)) a = a1;
	t[3] = (GLubyte)a;
}

}  // extern "C"
