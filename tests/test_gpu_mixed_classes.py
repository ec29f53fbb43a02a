"""Batch classes that mix textures of few and many random colours: the blocks of every texture against the oracle,
whatever the largest count of the class."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _texture(rng, w, h, kind):
    y, x = np.mgrid[0:h, 0:w]
    if kind == 0:  # small colour boxes
        a = np.stack([128 + 90 * np.sin(x / 37.0), 128 + 90 * np.cos(y / 41.0), 200 + 30 * np.sin((x + y) / 53.0)], 2)
        a = a + rng.integers(-3, 4, (h, w, 3))
    elif kind == 1:  # boxes of some tens of cells
        a = np.stack([128 + 90 * np.sin(x / 7.0), 128 + 90 * np.cos(y / 6.0), 128 + 80 * np.sin((x + y) / 8.0)], 2)
    else:
        a = rng.integers(0, 256, (h, w, 3))
    alpha = rng.integers(0, 256, (h, w, 1)) if kind == 2 else np.full((h, w, 1), 255)
    return np.concatenate([a, alpha], 2).clip(0, 255).astype(np.uint8).reshape(-1)


@pytest.mark.parametrize("cd", range(8))
def test_counts_of_one_class(gpu, oracle, cd):
    """8 to 112 random colours in one class: blocks with 2 to 8 row blocks share its kernel and group memory.  One
    size has more than 2048 tiles of four blocks, the other fewer."""
    rng = np.random.default_rng(40 + cd)
    for side, counts in ((101, (8, 1, 16, 32, 64)), (230, (8, 24, 112, 48, 17))):
        items = [dict(rgba=_texture(rng, side, side - 3 * i, i % 3), width=side, height=side - 3 * i, dxt=i % 3, cd=cd,
                      nrandom=n, refine=i % 3, seed=7 + i) for i, n in enumerate(counts)]
        imgs = gpu.DeviceImages(items)
        b = gpu.Batch(imgs)
        print(f"mixed class cd={cd} side={side} counts={counts}", flush=True)
        b.launch()
        gpu.synchronize()
        host = imgs.dst.to_host()
        for i, it in enumerate(items):
            q = oracle.rgb565_image(it["rgba"], it["width"], it["height"], 4, (1, 4, 8)[it["dxt"]], 0)
            exp = oracle.encode_quantized(q, it["width"], it["height"], it["dxt"], cd, it["nrandom"], it["refine"],
                                          it["seed"])
            assert np.array_equal(imgs.output(i, host), exp), (i, it["nrandom"])
        b.destroy()
        imgs.free()
