"""s2tc_amd_colordist_error over more tiles than workgroups, ragged edges, unaligned blocks and several threads at
once, against the oracle."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _case(gpu, oracle, rng, w, h, dxt, cd):
    q = np.stack([rng.integers(0, 32, w * h), rng.integers(0, 64, w * h), rng.integers(0, 32, w * h),
                  rng.integers(0, 2, w * h)], axis=1).astype(np.uint8).reshape(-1)
    blocks = rng.integers(0, 256, gpu.nblocks(w, h) * gpu.block_bytes(dxt)).astype(np.uint8)
    return q, blocks, oracle.colordist_error(q, w, h, dxt, cd, blocks)


# 256 x 16 texels a tile, at most 512 workgroups
@pytest.mark.parametrize("w,h,dxt,cd", [(256, 16, 0, 5), (255, 15, 2, 2), (257, 17, 1, 7), (2048, 1024, 0, 3),
                                        (2049, 1023, 2, 0), (300, 8209, 0, 1)])
def test_tiles(gpu, oracle, w, h, dxt, cd):
    q, blocks, exp = _case(gpu, oracle, np.random.default_rng(w + h), w, h, dxt, cd)
    print(f"colour-distance sum {w}x{h} dxt={dxt} cd={cd}", flush=True)
    assert gpu.colordist_error(q, w, h, blocks, dxt, cd) == exp
    d_q, d_b = gpu.DeviceBuffer.from_host(q), gpu.DeviceBuffer(blocks.size + 16)
    gpu.check(gpu.lib().s2tc_amd_memcpy_h2d(d_b.ptr + 3, blocks.ctypes.data, blocks.size))
    assert gpu.colordist_error_device(d_q, 0, w, h, d_b.ptr + 3, dxt, cd) == exp


def test_threads(gpu, oracle):
    cases = [(w, h, dxt, cd) + _case(gpu, oracle, np.random.default_rng(k), w, h, dxt, cd)
             for k, (w, h, dxt, cd) in enumerate([(64, 64, 0, 5), (500, 300, 2, 4), (1000, 17, 1, 6), (33, 700, 0, 0)])]
    bad = []

    def work(c):
        w, h, dxt, cd, q, blocks, exp = c
        for _ in range(8):
            if gpu.colordist_error(q, w, h, blocks, dxt, cd) != exp:
                bad.append(c[:4])

    print("colour-distance sums, 4 threads", flush=True)
    ts = [threading.Thread(target=work, args=(c,)) for c in cases]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
