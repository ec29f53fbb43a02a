"""s2tc_amd_mip_chain from a source that lies where the chain's smaller levels go (level 0 is copied before they are
written), against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(64, 64), (1000, 700), (2048, 2048)])
@pytest.mark.parametrize("at", [1, 2])
def test_source_over_the_levels(gpu, oracle, w, h, at):
    rgba = np.random.default_rng(w + at).integers(0, 256, w * h * 4).astype(np.uint8)
    layout, total = gpu.mip_layout(w, h)
    start = layout[at][0]
    print(f"mip chain {w}x{h}, source at level {at}", flush=True)
    d = gpu.DeviceBuffer(start + rgba.nbytes)
    gpu.check(gpu.lib().s2tc_amd_memcpy_h2d(d.ptr + start, rgba.ctypes.data, rgba.nbytes))
    assert gpu.mip_chain_device(d.ptr + start, w, h, d, total) == len(layout)
    gpu.synchronize()
    host = d.to_host(total)
    for (o, lw, lh), (ew, eh, lv) in zip(layout, oracle.mip_chain(rgba, w, h)):
        assert (lw, lh) == (ew, eh) and np.array_equal(host[o:o + lw * lh * 4], lv), (lw, lh)
