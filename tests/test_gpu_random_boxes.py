"""Random-candidate kernels on blocks whose colour boxes have every number of cells around the limits of the scan over
distinct colours (8 and 16 colours, the tables of each candidate count, 256 cells), whole and partial, with two and
three row blocks in registers (the latter from 49 to 112 random colours in more than 2048 workgroups)."""
import numpy as np
import pytest

import imgutil


def _boxes(rng, w, h):
    """Quantized texels (r5 g6 b5 a8); every block draws its colours and alphas from a small random box."""
    bh, bw = (h + 3) // 4, (w + 3) // 4
    out = np.zeros((4 * bh, 4 * bw, 4), np.int64)
    for c, top in enumerate((32, 64, 32, 256)):
        size = rng.choice([1, 1, 2, 2, 3, 4, 5, 8, 9, 16], (bh, bw))
        lo = (rng.random((bh, bw)) * (top - size + 1)).astype(int)
        up = lambda a: np.repeat(np.repeat(a, 4, 0), 4, 1)
        out[..., c] = up(lo) + (rng.random((4 * bh, 4 * bw)) * up(size)).astype(int)
    return np.ascontiguousarray(out[:h, :w].astype(np.uint8))


@pytest.mark.gpu
@pytest.mark.parametrize("cd", range(8))
@pytest.mark.parametrize("w,h,counts", [(66, 35, (1, 16, 17, 24, 32, 33, 48, 49, 112, 113, 208)),
                                        (513, 259, (49, 64, 112)), (1021, 130, (48, 80, 113))])
def test_small_boxes(gpu, oracle, cd, w, h, counts):
    rng = np.random.default_rng(900 + cd)
    for k, nr in enumerate(counts):
        dxt, refine = (k + cd) % 3, (k // 3 + cd) % 3
        q = _boxes(rng, w, h)
        if dxt == 0:
            q[..., 3] = rng.random((h, w)) < 0.9
        elif dxt == 1:
            q[..., 3] &= 15
        print(f"boxes cd={cd} {w}x{h} dxt={dxt} nrandom={nr} refine={refine}", flush=True)
        exp = oracle.encode_quantized(q.reshape(-1), w, h, dxt, cd, nr, refine, 5)
        d_s = gpu.DeviceBuffer.from_host(q)
        d_o = gpu.DeviceBuffer(exp.size)
        gpu.encode_image_device(d_s.ptr, 0, w, h, d_o.ptr, dxt, cd, nr, refine, 5)
        gpu.synchronize()
        assert np.array_equal(d_o.to_host(), exp), (w, h, dxt, nr, refine)
        imgs = gpu.DeviceImages([dict(rgba=q.reshape(-1), width=w, height=h, dxt=dxt, cd=cd, nrandom=nr, refine=refine,
                                      seed=5)], src_kind=gpu.SRC_QUANTIZED)
        b = gpu.Batch(imgs)
        b.launch()
        gpu.synchronize()
        out = imgs.dst.to_host()[imgs.dst_off[0]:][:exp.size]
        b.destroy()
        assert np.array_equal(out, exp), ("batch", w, h, dxt, nr, refine)


def _near(x):
    x = np.asarray(x, np.float32)
    return [x, np.nextafter(x, np.float32(np.inf)), np.nextafter(x, np.float32(-np.inf))]


def test_division_by_reciprocal_is_exact():
    """The arithmetic of the kernels' Mean (round-half-up mean of up to 16 values up to 255) and Modulo (31 bits by up
    to 256), with reciprocals one unit off either way."""
    for n in range(1, 17):
        s = np.arange(255 * n + 1)
        for rn in _near(np.float32(1) / np.float32(n)):
            got = np.floor(np.float32(s.astype(np.float64) * np.float64(rn) + 0.515625))
            assert np.array_equal(got.astype(int), ((s << 1) + n) // (n << 1)), n
    for l in range(1, 257):
        for r in _near(np.float32(1) / np.float32(l)):
            q = int(np.float32(r * np.float32(4294963200.0)))
            rem = ((1 << 32) - 1 - q * l) & 0xFFFFFFFF
            m = q + int(np.float32(np.float64(rem) * np.float64(r) - 0.0009765625))
            assert (1 << 32) - 2 * l <= m * l <= 1 << 32 and m < 1 << 32, (l, m)
            k = np.unique(np.concatenate([np.arange(0, 3000), np.random.default_rng(l).integers(0, 1 << 31, 3000)]) // l)
            x = np.concatenate([k * l, k * l + l - 1, [2 ** 31 - 1]]).astype(np.uint64)
            x = x[x < 1 << 31]
            hi = (x * np.uint64(m)) >> np.uint64(32)
            rr = (x - (hi & np.uint64(0xFFFFFF)) * np.uint64(l)) & np.uint64(0xFFFFFF)
            rr = np.where(rr >= l, rr - np.uint64(l), rr)
            assert np.array_equal(rr, x % np.uint64(l)), l
