"""The launch forms of the Floyd-Steinberg dither that wide and tall images reach, against the oracle: carries in more
than 64 KiB of LDS (rows of 5369 to 13,216 texels), carries in memory alone (wider rows), and slabs whose rows have all
stretches of a wave's steps.  On the CPU, the quantizer's steps as the kernel writes them."""
import ctypes

import numpy as np
import pytest


def test_kernel_quantizer_exact():
    """floor(med3(fma(u, scale, bias), 0, maxv)) and floor(fma(q, deq, -2048)) of u = v - 2048 equal the 12-bit levels
    and the integer division by maxval, for every |v| < 2^18."""
    for shift in (2, 3, 4, 7):
        maxval = (1 << (8 - shift)) - 1
        scale = 2.0 ** -(shift + 4)
        deq = np.float32(4095.0 / maxval)
        if float(deq) < 4095.0 / maxval:
            deq = np.nextafter(deq, np.float32(8192))
        v = np.arange(-(1 << 18), 1 << 18, dtype=np.float64)
        # both fmas are exact in float64 and round once to float32
        level = np.floor(np.clip(((v - 2048) * scale + 2048 * scale).astype(np.float32), 0, maxval)).astype(int)
        assert np.array_equal(level, np.clip(v.astype(int) >> (shift + 4), 0, maxval)), shift
        q = np.arange(maxval + 1)
        back = np.floor((q.astype(np.float64) * float(deq) - 2048.0).astype(np.float32)).astype(int)
        assert np.array_equal(back, q * 4095 // maxval - 2048), shift


def _check(gpu, oracle, w, h, sc, ab, seed):
    L = gpu.lib()
    L.rgb565_image.argtypes = [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int] * 5
    print(f"FS dither {w}x{h} srccomps={sc} alphabits={ab}", flush=True)
    src = np.random.default_rng(seed).integers(0, 256, w * h * sc, dtype=np.uint8)
    out = np.zeros(w * h * 4, np.uint8)
    L.rgb565_image(out.ctypes.data, src.ctypes.data, w, h, sc, ab, 2)
    assert np.array_equal(out, oracle.rgb565_image(src, w, h, sc, ab, 2))


@pytest.mark.gpu
@pytest.mark.parametrize("w", [5360, 5368, 5369, 5376, 5377, 13215, 13216, 13217, 13225, 16384])
def test_wide_rows(gpu, oracle, w):
    for k, (sc, ab, h) in enumerate([(4, 1, 65), (4, 4, 130), (4, 8, 194), (3, 8, 64), (4, 1, 1)]):
        _check(gpu, oracle, w, h, sc, ab, w + k)


@pytest.mark.gpu
@pytest.mark.parametrize("w,h,ab", [(131, 232960 + 70, 4), (131, 232960 + 65, 1), (128, 262144 + 1, 8)])
def test_slabs_of_whole_stretches(gpu, oracle, w, h, ab):
    """Rows as wide as a wave's lag and more rows than a slab holds (232,960 and 262,144 at these widths)."""
    _check(gpu, oracle, w, h, 4, ab, h)
