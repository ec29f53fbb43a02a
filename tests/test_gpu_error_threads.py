"""s2tc_amd_colordist_error from several threads at once: equal to the oracle, and a thread's error fails the test."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_threads_and_their_errors(gpu, oracle):
    cases = []
    for k, (w, h, dxt, cd) in enumerate([(64, 64, 0, 5), (500, 300, 2, 4), (1000, 17, 1, 6), (33, 700, 0, 0)]):
        rng = np.random.default_rng(k)
        q = np.stack([rng.integers(0, 32, w * h), rng.integers(0, 64, w * h), rng.integers(0, 32, w * h),
                      rng.integers(0, 2, w * h)], axis=1).astype(np.uint8).reshape(-1)
        blocks = rng.integers(0, 256, gpu.nblocks(w, h) * gpu.block_bytes(dxt)).astype(np.uint8)
        cases.append((w, h, dxt, cd, q, blocks, oracle.colordist_error(q, w, h, dxt, cd, blocks)))

    def work(c):
        w, h, dxt, cd, q, blocks, exp = c
        for _ in range(8):
            assert gpu.colordist_error(q, w, h, blocks, dxt, cd) == exp, c[:4]

    print("colour-distance sums, 4 threads", flush=True)
    with ThreadPoolExecutor(4) as pool:
        for f in [pool.submit(work, c) for c in cases]:
            f.result()
        with pytest.raises(gpu.S2tcError):  # a width of 0 is refused, and the refusal reaches the caller
            pool.submit(gpu.colordist_error, cases[0][4], 0, 64, cases[0][5], 0, 5).result()
