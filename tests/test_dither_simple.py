"""The SIMPLE dither (s2tc_amd/csrc/dither.hip): the byte form of its state
transitions on the CPU, and the scan on the GPU against the oracle around the
sizes of its chunks, waves and workgroups."""
import ctypes

import numpy as np
import pytest


def _diffuse(v, d, sh):
    """diffuse() of s2tc_algorithm.cpp: the new error of source value v after error d."""
    s = v + d
    r = np.clip(s >> sh, 0, (1 << (8 - sh)) - 1)
    return s - ((r << sh) | (r >> (8 - 2 * sh)))


@pytest.mark.parametrize("sh", [2, 3, 4])
def test_byte_transitions_exact(sh):
    """SimpleMap::step for every source value and error: x = (d + OFF) + m, the new d + OFF is x mod OFF plus the table
    byte x / OFF, and no byte leaves 0 .. 2 OFF - 1."""
    off, last = 1 << sh, (1 << (8 - sh)) - 1
    for v in range(256):
        q, m = v >> sh, v & (off - 1)
        e = [off if q == 0 else (q - 1) >> (8 - 2 * sh), q >> (8 - 2 * sh), -1 if q == last else (q + 1) >> (8 - 2 * sh)]
        tab = np.array([off - k for k in e])
        assert tab.min() >= 0
        d = np.arange(-(off - 1), off)
        x = d + off + m
        new = (x & (off - 1)) + tab[x >> sh]
        assert np.array_equal(new - off, _diffuse(v, d, sh)), v
        assert new.min() >= 1 and new.max() < 2 * off
        x0 = m  # the byte of no state
        assert 0 <= (x0 & (off - 1)) + tab[x0 >> sh] < 2 * off


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 7, 8, 9, 63, 64, 65, 511, 512, 513, 2047, 8191, 8192, 8193, 32767, 32768, 32769, 65535,
                               65536, 65537, 131071, 131072, 131073, 139264, 139265, 1000003])
def test_chunks_and_scans(gpu, oracle, n):
    """Texel counts around the chunk lengths (8, 16, 32), the one-workgroup form (8192), the 64 waves that the emit
    kernel scans by itself (131072) and ragged ends, on noise, saturated noise, ramps and flat texels."""
    L = gpu.lib()
    L.rgb565_image.argtypes = [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int] * 5
    rng = np.random.default_rng(n)
    for kind in range(4):
        a = rng.integers(0, 256, (n, 4))
        if kind == 1:
            a = (a & 1) * 255
        if kind == 2:
            a = (np.arange(n)[:, None] * np.array([1, 3, 2, 5]) // 11) % 256
        if kind == 3:
            a = np.zeros((n, 4), int) + rng.integers(0, 256, 4)
        for sc, ab in ((4, 1), (4, 4), (4, 8), (3, 4)):
            print(f"SIMPLE dither n={n} kind={kind} srccomps={sc} alphabits={ab}", flush=True)
            src = np.ascontiguousarray(a[:, :sc].astype(np.uint8)).reshape(-1)
            out = np.zeros(n * 4, np.uint8)
            L.rgb565_image(out.ctypes.data, src.ctypes.data, n, 1, sc, ab, 1)
            assert np.array_equal(out, oracle.rgb565_image(src, n, 1, sc, ab, 1)), (n, kind, sc, ab)
