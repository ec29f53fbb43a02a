// Host checks of CopyCrew (staging.h), compiled with g++ by
// tests/test_copy_crew.py.  Prints "ok" and exits 0 when every check passes.
#include <time.h>

#include <chrono>
#include <cstdio>
#include <functional>
#include <numeric>

#include "staging.h"

using s2tc::CopyCrew;

static double cpu_seconds()
{
	timespec t;
	clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
	return (double)t.tv_sec + 1e-9 * (double)t.tv_nsec;
}

static void nap(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

static bool wait_for(const std::function<bool()> &done)
{
	for (int i = 0; i < 5000; ++i) {
		if (done()) return true;
		nap(1);
	}
	return false;
}

int main()
{
	const size_t chunk = 4096, n = 9 * chunk + 77, ring = 4;
	std::vector<uint8_t> src(n), stage(ring * chunk), blocks(1000 * 16), dest(1000 * 24, 0x5c);
	std::iota(src.begin(), src.end(), 0);
	std::iota(blocks.begin(), blocks.end(), 3);
	CopyCrew crew(src.data(), n, stage.data(), chunk, ring);
	crew.set_rows(dest.data(), blocks.data(), 16, 24, 1000);
	crew.start(3);

	// helpers with nothing to copy sleep: three that spin would take 3 x 400 ms
	nap(50);
	double c0 = cpu_seconds();
	nap(400);
	if (cpu_seconds() - c0 > 0.1) {
		printf("idle helpers took %.3f s of CPU time in 0.4 s\n", cpu_seconds() - c0);
		return 1;
	}
	// they wake up for chunks and for rows, by themselves, every time
	for (size_t i = 0; i < crew.nchunks; ++i) {
		if (i % 3 == 0) nap(20);
		crew.open_chunks(i + 1);
		if (!wait_for([&] { return crew.chunk_copied(i); })) {
			printf("chunk %zu was not copied\n", i);
			return 1;
		}
		if (memcmp(stage.data() + crew.ring_offset(i), src.data() + i * chunk, crew.chunk_len(i))) {
			printf("chunk %zu is wrong\n", i);
			return 1;
		}
	}
	nap(50);
	crew.open_rows(1000);
	if (!wait_for([&] { return crew.rows_copied(); })) {
		printf("rows were not copied\n");
		return 1;
	}
	for (int r = 0; r < 1000; ++r)
		if (memcmp(&dest[24 * r], &blocks[16 * r], 16) || dest[24 * r + 16] != 0x5c) {
			printf("row %d is wrong\n", r);
			return 1;
		}
	// and sleep again
	nap(50);
	c0 = cpu_seconds();
	nap(200);
	if (cpu_seconds() - c0 > 0.05) {
		printf("helpers without work took %.3f s of CPU time in 0.2 s\n", cpu_seconds() - c0);
		return 1;
	}
	// many short calls: none hangs, whichever side is first
	for (int k = 0; k < 300; ++k) {
		CopyCrew c(src.data(), n, stage.data(), chunk, ring);
		c.start(k % 4);
		size_t open = ring;
		c.open_chunks(open);
		for (size_t i = 0; i < c.nchunks; ++i) {
			while (!c.chunk_copied(i))
				if (!c.step()) std::this_thread::yield();
			if (open < c.nchunks) c.open_chunks(++open);
			if (k % 50 == 0) nap(1);
		}
	}
	printf("ok\n");
	return 0;
}
