"""tx_compress_dxtn around the sizes where the way of its host data changes (512 KiB read in place, 1 MiB in one
piece, 8 MiB in bands), with row gaps, few rows, and a destination over the source, against the oracle."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NAMES = ["RGB", "YUV", "SRGB", "SRGB_MIXED", "AVG", "WAVG", "W0AVG", "NORMALMAP"]
DITHERS = ["NONE", "SIMPLE", "FLOYDSTEINBERG"]


@pytest.fixture
def call(gpu, oracle, monkeypatch):
    L = gpu.lib()
    L.tx_compress_dxtn.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_uint,
                                   ctypes.c_void_p, ctypes.c_int]
    L.tx_compress_dxtn.restype = None

    def run(sc, w, h, fmt, dither, cd=5, nr=-1, gap=0, in_place=False):
        for k, v in dict(DITHER_MODE=DITHERS[dither], COLORDIST_MODE=NAMES[cd], RANDOM_COLORS=str(nr),
                         REFINE_COLORS="ALWAYS", RANDOM_SEED="3").items():
            monkeypatch.setenv("S2TC_" + k, v)
        bs = 8 if fmt < 0x83F2 else 16
        bw, bh = (w + 3) // 4, (h + 3) // 4
        rng = np.random.default_rng(w + 7 * h + sc + fmt)
        src = rng.integers(0, 256, w * h * sc).astype(np.uint8)
        print(f"call {w}x{h}x{sc} {fmt:#x} {DITHERS[dither]} cd={cd} nrandom={nr} gap={gap} in_place={in_place}",
              flush=True)
        r, exp = oracle.compress(sc, w, h, src, fmt, bw * bs, cd, nr, 1, dither, 3)
        exp = exp[:bw * bh * bs].reshape(bh, bw * bs)
        stride = bw * bs + gap
        dst = src if in_place else np.full(stride * bh + 64, 0x5C, np.uint8)
        L.tx_compress_dxtn(sc, w, h, src.ctypes.data, fmt, dst.ctypes.data, stride)
        rows = dst[:stride * bh].reshape(bh, stride)
        assert np.array_equal(rows[:, :bw * bs], exp)
        if not in_place:
            assert (rows[:, bw * bs:] == 0x5C).all() and (dst[stride * bh:] == 0x5C).all()

    return run


@pytest.mark.parametrize("dither", [0, 1, 2])
@pytest.mark.parametrize("sc,w,h", [(4, 512, 256), (4, 513, 256), (4, 1023, 256), (4, 1025, 256), (3, 701, 499),
                                    (4, 2047, 1024), (4, 2047, 1026), (3, 2799, 1001)])
def test_sizes(call, sc, w, h, dither):
    call(sc, w, h, 0x83F1 if w & 1 else 0x83F3, dither, gap=0 if h & 2 else 48)


@pytest.mark.parametrize("fmt", [0x83F0, 0x83F2, 0x83F3])
@pytest.mark.parametrize("sc,w,h", [(4, 129, 65), (3, 129, 65), (3, 400, 437), (4, 361, 363)])
def test_simple_from_pinned_memory(call, sc, w, h, fmt):
    call(sc, w, h, fmt, 1)


@pytest.mark.parametrize("sc,w,h,dither", [(4, 300001, 7, 1), (4, 240001, 9, 1), (3, 300000, 10, 0), (4, 120001, 19, 0),
                                           (4, 5, 500001, 1)])
def test_bands_of_extreme_shapes(call, sc, w, h, dither):
    call(sc, w, h, 0x83F0, dither, nr=0 if h == 9 else -1)


@pytest.mark.parametrize("w,h", [(64, 64), (1024, 512), (1535, 1537)])
def test_destination_over_the_source(call, w, h):
    call(4, w, h, 0x83F3, 1, in_place=True)
    call(4, w, h, 0x83F1, 0, in_place=True)
