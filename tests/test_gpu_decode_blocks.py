"""k_decode's lane per block: widths around a block and a wave's 64 blocks, and block and texel buffers that are only
as aligned as bytes and texels are, against the oracle's decode."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", [0x83F0, 0x83F1, 0x83F2, 0x83F3])
def test_decode_edges_and_alignment(gpu, oracle, fmt):
    rng = np.random.default_rng(fmt)
    bs = 8 if fmt in (0x83F0, 0x83F1) else 16
    for w in (1, 2, 3, 4, 5, 255, 256, 257, 259):
        for h in (1, 3, 4, 17):
            nb = gpu.nblocks(w, h)
            blocks = rng.integers(0, 256, (nb, bs)).astype(np.uint8)
            blocks[::3, 0] = 0  # DXT5 alphas in the 6-value mode
            for off_b, off_t in ((0, 0), (1, 4), (8, 12), (6, 8)):
                print(f"decode fmt={fmt:#x} {w}x{h} blocks at +{off_b}, texels at +{off_t}", flush=True)
                d_b = gpu.DeviceBuffer(nb * bs + 64)
                d_t = gpu.DeviceBuffer(w * h * 4 + 64)
                host = np.zeros(nb * bs + 64, np.uint8)
                host[off_b:off_b + nb * bs] = blocks.reshape(-1)
                gpu.check(gpu.lib().s2tc_amd_memcpy_h2d(d_b.ptr, host.ctypes.data, host.size))
                d_t.fill(0xAB)
                gpu.decode_image_device(d_b.ptr + off_b, fmt, w, h, d_t.ptr + off_t)
                gpu.synchronize()
                out = d_t.to_host()
                exp = oracle.decode_image(blocks.reshape(-1), fmt, w, h)
                assert np.array_equal(out[off_t:off_t + w * h * 4], exp), (fmt, w, h, off_b)
                assert (out[:off_t] == 0xAB).all() and (out[off_t + w * h * 4:] == 0xAB).all()
