// staging.h - host threads between a caller's pageable buffers and pinned memory.
#pragma once

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace s2tc {

// Byte range [lo, hi) of a len-byte chunk that host thread t of nt copies
// into pinned staging.  Slices are whole 64-byte lines of ceil(len / nt)
// bytes rounded up, so nt of them reach at least len: together they cover
// [0, len) without overlap; trailing slices may be short or empty.
inline void stage_slice(size_t len, unsigned nt, unsigned t, size_t &lo, size_t &hi)
{
	const size_t per = ((len + nt - 1) / nt + 63) & ~(size_t)63;
	lo = std::min(len, per * t);
	hi = std::min(len, lo + per);
}

// The copies of one call, split into slices that the calling thread and its
// helpers take one by one: first those of the source (chunks of `chunk` bytes
// into a ring of `ring` pinned buffers), then those of the block rows that came
// back.  A slice can only be taken once its chunk or its rows are opened by the
// calling thread, which alone talks to the GPU.  Helpers that find no open slice
// for a while sleep until one is opened: a call may wait long for its encoder.
struct CopyCrew {
	static const unsigned kParts = 8;  // slices per chunk
	// Unsuccessful looks (about 50 us of yields, two chunks' uploads) before a
	// helper sleeps; waking one takes about as long.
	static const unsigned kIdle = 128;

	const uint8_t *src;
	uint8_t *stage;
	const size_t n, chunk, nchunks, ring;
	std::unique_ptr<std::atomic<unsigned>[]> done;  // copied slices of each chunk
	std::atomic<size_t> up_next{0}, up_open{0};     // slices

	uint8_t *dest = nullptr;
	const uint8_t *blocks = nullptr;
	size_t row_bytes = 0, row_pitch = 0;
	int nrows = 0, rows_per_slice = 1;
	std::atomic<size_t> out_next{0}, out_open{0}, out_done{0};

	std::atomic<bool> quit{false};
	std::atomic<unsigned> asleep{0};
	std::mutex mu;
	std::condition_variable opened;
	std::vector<std::thread> helpers;

	CopyCrew(const uint8_t *src_, size_t n_, uint8_t *stage_, size_t chunk_, size_t ring_)
	    : src(src_), stage(stage_), n(n_), chunk(chunk_), nchunks((n_ + chunk_ - 1) / chunk_), ring(ring_),
	      done(new std::atomic<unsigned>[nchunks])
	{
		for (size_t i = 0; i < nchunks; ++i) done[i].store(0, std::memory_order_relaxed);
	}
	~CopyCrew() { finish(); }
	CopyCrew(const CopyCrew &) = delete;
	CopyCrew &operator=(const CopyCrew &) = delete;

	// Rows of finished blocks go to dest (rows that do not overlap).
	void set_rows(uint8_t *dest_, const uint8_t *blocks_, size_t row_bytes_, size_t row_pitch_, int nrows_)
	{
		dest = dest_;
		blocks = blocks_;
		row_bytes = row_bytes_;
		row_pitch = row_pitch_;
		nrows = nrows_;
		rows_per_slice = (int)std::max((size_t)1, ((size_t)256 << 10) / row_bytes);
	}
	size_t out_slices() const { return ((size_t)nrows + rows_per_slice - 1) / rows_per_slice; }

	// Starts up to `count` helpers; with fewer (or none) the call is only slower.
	void start(unsigned count)
	{
		try {
			helpers.reserve(count);
			for (unsigned t = 0; t < count; ++t)
				helpers.emplace_back([this] { help(); });
		} catch (const std::exception &) {
		}
	}
	void finish()
	{
		quit.store(true);
		wake();
		for (auto &h : helpers) h.join();
		helpers.clear();
	}

	size_t ring_offset(size_t i) const { return i % ring * chunk; }
	size_t chunk_len(size_t i) const { return std::min(chunk, n - i * chunk); }
	// chunks before `i` may be copied (their buffers are free)
	void open_chunks(size_t i)
	{
		up_open.store(i * kParts);
		wake();
	}
	bool chunk_copied(size_t i) const { return done[i].load(std::memory_order_acquire) == kParts; }
	// block rows before `rows` have come back
	void open_rows(int rows)
	{
		out_open.store(rows >= nrows ? out_slices() : (size_t)(rows / rows_per_slice));
		wake();
	}
	bool rows_copied() const { return out_done.load(std::memory_order_acquire) == out_slices(); }

	// Copies one open slice; false if there is none.
	bool step()
	{
		size_t i;
		if (take(up_next, up_open, i)) {
			const size_t c = i / kParts;
			size_t lo, hi;
			stage_slice(chunk_len(c), kParts, (unsigned)(i % kParts), lo, hi);
			if (hi > lo) memcpy(stage + ring_offset(c) + lo, src + c * chunk + lo, hi - lo);
			done[c].fetch_add(1, std::memory_order_release);
			return true;
		}
		if (take(out_next, out_open, i)) {
			const int r0 = (int)i * rows_per_slice, r1 = std::min(nrows, r0 + rows_per_slice);
			for (int r = r0; r < r1; ++r)
				memcpy(dest + (size_t)r * row_pitch, blocks + (size_t)r * row_bytes, row_bytes);
			out_done.fetch_add(1, std::memory_order_release);
			return true;
		}
		return false;
	}

private:
	bool has_work() const { return quit.load() || up_next.load() < up_open.load() || out_next.load() < out_open.load(); }
	// A helper counts itself asleep before it looks for work the last time, and
	// whoever opens slices looks for sleepers afterwards, both in the one order of
	// the sequentially consistent operations: one of the two sees the other.
	void wake()
	{
		if (!asleep.load()) return;
		std::lock_guard<std::mutex> lk(mu);
		opened.notify_all();
	}
	void help()
	{
		unsigned idle = 0;
		while (!quit.load(std::memory_order_acquire)) {
			if (step()) {
				idle = 0;
			} else if (++idle < kIdle) {
				std::this_thread::yield();
			} else {
				std::unique_lock<std::mutex> lk(mu);
				++asleep;
				opened.wait(lk, [this] { return has_work(); });
				--asleep;
				idle = 0;
			}
		}
	}
	static bool take(std::atomic<size_t> &next, const std::atomic<size_t> &open, size_t &i)
	{
		i = next.load(std::memory_order_relaxed);
		while (i < open.load(std::memory_order_acquire))
			if (next.compare_exchange_weak(i, i + 1, std::memory_order_relaxed)) return true;
		return false;
	}
};

}  // namespace s2tc
