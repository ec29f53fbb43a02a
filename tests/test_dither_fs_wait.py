"""A wait of the Floyd-Steinberg dither that ends without what it waited for is an error of the call, not a wrong image
in silence.  The bound of the waits is lowered from the host: a wave then looks once and gives up, and every wave ends
as usual."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def lib(gpu):
    L = gpu.lib()
    L.rgb565_image.argtypes = [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int] * 5
    L.tx_compress_dxtn.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_uint,
                                   ctypes.c_void_p, ctypes.c_int]
    L.tx_compress_dxtn.restype = None
    L.s2tc_amd_debug_set_fs_polls.argtypes = [ctypes.c_uint]
    L.s2tc_amd_debug_set_fs_polls.restype = None
    yield L
    L.s2tc_amd_debug_set_fs_polls(0xFFFFFFFF)


def _dither(L, src, w, h, ab):
    out = np.zeros(w * h * 4, np.uint8)
    L.rgb565_image(out.ctypes.data, src.ctypes.data, w, h, 4, ab, 2)
    return out


# several bands: carries through LDS alone, and through LDS and memory
@pytest.mark.parametrize("w,h,ab", [(300, 130, 8), (700, 600, 1), (13300, 70, 8)])
def test_dither_that_stops_waiting(lib, oracle, capfd, w, h, ab):
    src = np.random.default_rng(w).integers(0, 256, w * h * 4).astype(np.uint8)
    exp = oracle.rgb565_image(src, w, h, 4, ab, 2)
    print(f"FS dither {w}x{h} alphabits={ab}, no waits", flush=True)
    lib.s2tc_amd_debug_set_fs_polls(0)
    _dither(lib, src, w, h, ab)
    assert "rgb565_image failed" in capfd.readouterr().err
    lib.s2tc_amd_debug_set_fs_polls(0xFFFFFFFF)
    assert np.array_equal(_dither(lib, src, w, h, ab), exp)
    assert "failed" not in capfd.readouterr().err


def test_encode_that_stops_waiting(lib, oracle, capfd, monkeypatch):
    monkeypatch.setenv("S2TC_DITHER_MODE", "FLOYDSTEINBERG")
    for k in ("COLORDIST_MODE", "RANDOM_COLORS", "REFINE_COLORS"):
        monkeypatch.delenv("S2TC_" + k, raising=False)
    w, h = 500, 300
    src = np.random.default_rng(1).integers(0, 256, w * h * 4).astype(np.uint8)
    dst = np.full(w * h, 0x5C, np.uint8)
    print(f"tx_compress_dxtn {w}x{h} FLOYDSTEINBERG, no waits", flush=True)
    lib.s2tc_amd_debug_set_fs_polls(0)
    lib.tx_compress_dxtn(4, w, h, src.ctypes.data, 0x83F3, dst.ctypes.data, 0)
    assert "tx_compress_dxtn failed" in capfd.readouterr().err
    assert (dst == 0x5C).all()
    lib.s2tc_amd_debug_set_fs_polls(0xFFFFFFFF)
    lib.tx_compress_dxtn(4, w, h, src.ctypes.data, 0x83F3, dst.ctypes.data, 0)
    r, exp = oracle.compress(4, w, h, src, 0x83F3, 0, 5, -1, 1, 2, 0)
    assert np.array_equal(dst, exp[:w * h])
