"""The Floyd-Steinberg dither of images of a few texels, which one wave does in one launch, around the largest of them,
against the oracle."""
import ctypes

import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("sc,ab", [(4, 1), (4, 4), (4, 8), (3, 1), (3, 8)])
def test_small_images(gpu, oracle, sc, ab):
    L = gpu.lib()
    L.rgb565_image.argtypes = [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int] * 5
    rng = np.random.default_rng(sc + ab)
    print(f"small FS dithers srccomps={sc} alphabits={ab}", flush=True)
    for w, h in [(w, h) for w in range(1, 41) for h in range(1, 41) if w * h <= 40]:
        for kind in range(2):
            src = (rng.integers(0, 256, w * h * sc) if kind == 0 else rng.integers(0, 2, w * h * sc) * 255).astype(np.uint8)
            out = np.zeros(w * h * 4, np.uint8)
            L.rgb565_image(out.ctypes.data, src.ctypes.data, w, h, sc, ab, 2)
            assert np.array_equal(out, oracle.rgb565_image(src, w, h, sc, ab, 2)), (w, h, kind)
