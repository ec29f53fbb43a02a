"""k_mip_levels: chains around the 64 x 64 tile and the six levels of a launch, from another buffer and in place,
against the oracle's Image_MipReduce32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(2, 2), (63, 65), (64, 64), (65, 63), (66, 66), (127, 129), (128, 1), (1, 128), (1, 4097),
                                 (4097, 1), (4095, 3), (2, 130), (191, 193), (8200, 70), (70, 8200), (4096, 64)])
def test_chain_tiles_and_launches(gpu, oracle, w, h):
    rng = np.random.default_rng(w * 10007 + h)
    rgba = rng.integers(0, 256, w * h * 4).astype(np.uint8)
    layout, total = gpu.mip_layout(w, h)
    exp = oracle.mip_chain(rgba, w, h)
    for in_place in (False, True):
        print(f"mip chain {w}x{h} in_place={in_place}", flush=True)
        d = gpu.DeviceBuffer(total)
        d.fill(0xAB)
        if in_place:
            gpu.check(gpu.lib().s2tc_amd_memcpy_h2d(d.ptr, rgba.ctypes.data, rgba.nbytes))
            src = d
        else:
            src = gpu.DeviceBuffer.from_host(rgba)
        assert gpu.mip_chain_device(src, w, h, d, total) == len(layout) == len(exp)
        gpu.synchronize()
        host = d.to_host(total)
        end = 0
        for (o, lw, lh), (ew, eh, lv) in zip(layout, exp):
            assert (host[end:o] == 0xAB).all()  # nothing between the levels
            assert (lw, lh) == (ew, eh) and np.array_equal(host[o:o + lw * lh * 4], lv), (lw, lh)
            end = o + lw * lh * 4
