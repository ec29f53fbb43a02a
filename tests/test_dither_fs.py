"""The Floyd-Steinberg dither (s2tc_amd/csrc/dither_fs.hip): its fp32 forms of
the reference's integer divisions on the CPU, and the wavefront on the GPU
against the oracle around the sizes of its bands, slots and slabs."""
import ctypes

import numpy as np
import pytest


def _fma32(a, b, c):
    """fmaf: the product of a value below 2^20 and a float, plus a float, is exact in float64."""
    return (a.astype(np.float64) * float(np.float32(b)) + float(np.float32(c))).astype(np.float32)


def _cdiv(a, b):
    return np.sign(a) * (np.abs(a) // b)


def test_split_divisions_exact():
    """trunc(fma) equals the C divisions of floyd (s2tc_algorithm.cpp:1227-1233) for every error below 2^18."""
    e = np.arange(-(1 << 18), 1 << 18, dtype=np.int64)
    assert np.array_equal(np.trunc(_fma32(e, 0.4375, 0.5)).astype(np.int64), _cdiv(e * 7 + 8, 16))
    assert np.array_equal(np.trunc(_fma32(e, 0.333333343, 0.444444448)).astype(np.int64), _cdiv(e * 3 + 4, 9))
    assert np.array_equal(np.trunc(_fma32(e, 0.833333373, 0.5)).astype(np.int64), _cdiv(e * 5 + 3, 6))


def test_quantizer_steps_exact():
    """q * 4095 / maxval as trunc(q * deq), deq the float at or above 4095 / maxval, and the 12-bit levels as
    floor(v * 2^-k) clamped."""
    for shift in (2, 3, 4, 7):
        maxval = (1 << (8 - shift)) - 1
        deq = np.float32(4095.0 / maxval)
        if float(deq) < 4095.0 / maxval:
            deq = np.nextafter(deq, np.float32(8192))
        q = np.arange(maxval + 1)
        assert np.array_equal(np.trunc(q.astype(np.float32) * deq).astype(int), q * 4095 // maxval), shift
        v = np.arange(-(1 << 18), 1 << 18)
        f = np.floor(np.clip(v.astype(np.float32) * np.float32(2.0 ** -(shift + 4)), 0, maxval)).astype(int)
        assert np.array_equal(f, np.clip(v >> (shift + 4), 0, maxval)), shift


def _dither(gpu, src, w, h, sc, ab):
    L = gpu.lib()
    L.rgb565_image.argtypes = [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int] * 5
    out = np.zeros(w * h * 4, np.uint8)
    L.rgb565_image(out.ctypes.data, src.ctypes.data, w, h, sc, ab, 2)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("h", [1, 2, 63, 64, 65, 128, 129, 191])
def test_bands_and_slots(gpu, oracle, h):
    """Rows around the 64-row bands (an even and an odd last row feed the alpha pass differently) and widths around
    the 8-step slots and the 126-step lag, on noise, on saturated noise and on smooth texels."""
    rng = np.random.default_rng(h)
    for w in (1, 2, 7, 8, 9, 64, 125, 126, 127, 128, 135, 300):
        for kind in range(3):
            n = w * h
            a = rng.integers(0, 256, (n, 4))
            if kind == 1:
                a = (a & 1) * 255
            if kind == 2:
                a = (np.arange(n)[:, None] * np.array([1, 3, 2, 1]) // 7 + 100) % 256
            for sc, ab in ((4, 1), (4, 4), (4, 8), (3, 1)):
                print(f"FS dither {w}x{h} kind={kind} srccomps={sc} alphabits={ab}", flush=True)
                src = np.ascontiguousarray(a[:, :sc].astype(np.uint8)).reshape(-1)
                assert np.array_equal(_dither(gpu, src, w, h, sc, ab), oracle.rgb565_image(src, w, h, sc, ab, 2)), (
                    w, h, kind, sc, ab)


@pytest.mark.gpu
def test_several_slabs(gpu, oracle):
    """An image of more rows than one slab of planes holds (419,392 at this width): the carries cross the slabs, and
    the alpha pass runs after the last one."""
    w, h = 3, 420000
    rng = np.random.default_rng(5)
    src = rng.integers(0, 256, w * h * 4).astype(np.uint8)
    for ab in (1, 8):
        print(f"FS dither {w}x{h} alphabits={ab}", flush=True)
        assert np.array_equal(_dither(gpu, src, w, h, 4, ab), oracle.rgb565_image(src, w, h, 4, ab, 2)), ab
