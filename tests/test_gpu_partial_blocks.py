"""Quick mode on images whose partial blocks run beside the full ones, on their own (none are full, or tall and narrow
images: more than 500 rows of workgroups of them), and whose block rows need two launches, against the oracle."""
import numpy as np
import pytest

import imgutil

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cd", [1, 2, 5])
@pytest.mark.parametrize("w,h,dxt,refine", [(1021, 515, 0, 2), (1023, 4, 2, 1), (4, 1023, 1, 0), (3, 2051, 2, 2),
                                            (2051, 3, 0, 1), (5, 512004, 0, 1), (5, 512005, 2, 0), (6, 1040009, 0, 2),
                                            (8, 1040004, 0, 1)])
def test_partial_blocks(gpu, oracle, cd, w, h, dxt, refine):
    rng = np.random.default_rng(w + h + cd)
    rgba = rng.integers(0, 256, w * h * 4).astype(np.uint8)
    q = oracle.rgb565_image(rgba, w, h, 4, imgutil.ALPHABITS[dxt], 0)
    exp = oracle.encode_quantized(q, w, h, dxt, cd, -1, refine, 3)
    for raw, src in ((1, rgba), (0, q)):
        print(f"partial blocks cd={cd} {w}x{h} dxt={dxt} refine={refine} raw={raw}", flush=True)
        d_s = gpu.DeviceBuffer.from_host(np.asarray(src).reshape(-1))
        d_o = gpu.DeviceBuffer(exp.size + 16)
        d_o.fill(0xAB)
        gpu.encode_image_device(d_s.ptr, raw, w, h, d_o.ptr, dxt, cd, -1, refine, 3)
        gpu.synchronize()
        out = d_o.to_host()
        assert np.array_equal(out[:exp.size], exp)
        assert (out[exp.size:] == 0xAB).all()
