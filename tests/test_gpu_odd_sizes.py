"""Quick mode and MODE_NORMAL on widths and heights that no block divides, from sources that are only as aligned as
their texels: the full blocks of k_fast_interior beside the partial ones, against the oracle."""
import numpy as np
import pytest

import imgutil

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cd", range(8))
def test_odd_sizes_and_sources(gpu, oracle, cd):
    rng = np.random.default_rng(70 + cd)
    for k, (w, h) in enumerate([(1, 9), (9, 1), (3, 3), (4, 5), (5, 4), (6, 1027), (257, 18), (1030, 7), (259, 261)]):
        for dxt in range(3):
            refine = (k + dxt) % 3
            nr = 0 if k % 3 == 2 else -1
            rgba = imgutil.smooth_rgba8(rng, w, h) if k % 2 else rng.integers(0, 256, w * h * 4).astype(np.uint8)
            q = oracle.rgb565_image(rgba, w, h, 4, imgutil.ALPHABITS[dxt], 0)
            exp = oracle.encode_quantized(q, w, h, dxt, cd, nr, refine, 3)
            for raw, src, off in ((1, rgba, 4), (0, q, 12)):
                print(f"odd size cd={cd} {w}x{h} dxt={dxt} refine={refine} nrandom={nr} raw={raw} +{off}", flush=True)
                host = np.zeros(w * h * 4 + 32, np.uint8)
                host[off:off + w * h * 4] = np.asarray(src).reshape(-1)
                d_s = gpu.DeviceBuffer.from_host(host)
                d_o = gpu.DeviceBuffer(exp.size + 16)
                d_o.fill(0xAB)
                gpu.encode_image_device(d_s.ptr + off, raw, w, h, d_o.ptr, dxt, cd, nr, refine, 3)
                gpu.synchronize()
                out = d_o.to_host()
                assert np.array_equal(out[:exp.size], exp), (w, h, dxt, refine, nr, raw)
                assert (out[exp.size:] == 0xAB).all()
