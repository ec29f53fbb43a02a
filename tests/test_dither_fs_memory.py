"""Device memory of the Floyd-Steinberg dither: with less scratch than an image takes it runs in smaller slabs with the
same result, and a large image's scratch is given back after the call."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MAX = ctypes.c_size_t(-1).value


@pytest.fixture
def lib(gpu):
    L = gpu.lib()
    L.rgb565_image.argtypes = [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int] * 5
    L.s2tc_amd_debug_set_fs_scratch_max.argtypes = [ctypes.c_size_t]
    L.s2tc_amd_debug_set_fs_scratch_max.restype = None
    yield L
    L.s2tc_amd_debug_set_fs_scratch_max(MAX)


def _dither(L, src, w, h, sc, ab):
    out = np.zeros(w * h * 4, np.uint8)
    L.rgb565_image(out.ctypes.data, src.ctypes.data, w, h, sc, ab, 2)
    return out


# a band of 64 rows takes 512 bytes a column and 80 KiB
@pytest.mark.parametrize("w,h,bands", [(300, 400, 1), (300, 513, 2), (131, 700, 3), (40, 1000, 5), (14000, 200, 2)])
def test_less_scratch(lib, oracle, capfd, w, h, bands):
    band = 4 * 64 * 16 * (((w + 7) // 8 + 16 + 3) // 4 * 4)
    for sc, ab in ((4, 1), (4, 4), (4, 8), (3, 8)):
        src = np.random.default_rng(w + ab).integers(0, 256, w * h * sc, dtype=np.uint8)
        print(f"FS dither {w}x{h} srccomps={sc} alphabits={ab}, scratch for {bands} bands", flush=True)
        lib.s2tc_amd_debug_set_fs_scratch_max(bands * band + 40 * w + (64 << 10))
        out = _dither(lib, src, w, h, sc, ab)
        assert "failed" not in capfd.readouterr().err
        assert np.array_equal(out, oracle.rgb565_image(src, w, h, sc, ab, 2)), (sc, ab)


def test_less_than_a_band(lib, capfd):
    src = np.zeros(300 * 100 * 4, np.uint8)
    print("FS dither 300x100, scratch for less than a band", flush=True)
    lib.s2tc_amd_debug_set_fs_scratch_max(100 << 10)
    _dither(lib, src, 300, 100, 4, 8)
    assert "rgb565_image failed" in capfd.readouterr().err
    lib.s2tc_amd_debug_set_fs_scratch_max(MAX)
    _dither(lib, src, 300, 100, 4, 8)
    assert "failed" not in capfd.readouterr().err


def _free_memory():
    hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so")  # the runtime that the library has loaded
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_large_scratch_is_given_back(lib, oracle):
    w, h = 8192, 5000  # planes of 320 MiB
    src = np.random.default_rng(3).integers(0, 256, w * h * 3, dtype=np.uint8)
    print(f"FS dither {w}x{h}, memory after the call", flush=True)
    _dither(lib, src[:3 * 64 * 64], 64, 64, 3, 8)
    free = _free_memory()
    out = _dither(lib, src, w, h, 3, 8)
    kept = free - _free_memory()
    # the context keeps the source and the result, as before there were planes
    assert kept < w * h * 7 + (64 << 20), kept
    assert np.array_equal(out, oracle.rgb565_image(src, w, h, 3, 8, 2))
