"""Performance cases: the calls that a user of this library makes, over the sizes they make them at.

Every case is one pass through a public entry point (the C ABI of
libtxc_dxtn.so or its Python view), from the smallest mip level that a GL
driver hands to tx_compress_dxtn to a 16384 x 16384 image on the device:

  txc     tx_compress_dxtn on host buffers, as a GL driver or the CLI calls it
  encode  one image that is already on the device
  batch   many textures with their mip chains in one graph launch
  decode  blocks on the device back to RGBA8
  error   total colour distance of an encoding (quality checks)
  mip     a full mip chain on the device
  s3tc    S3TC blocks remapped to S2TC on the device

A case is a dict of plain values; draw() gives more of the same ranges.
All outputs are bytes or whole numbers, so exact() has no value to give.
"""
import ctypes
import math
import os
from types import SimpleNamespace

import numpy as np
import torch

import s2tc_amd as s2
from s2tc_amd import synth, workloads

GL_FORMATS = {s2.DXT1: s2.GL_DXT1_RGBA, s2.DXT3: s2.GL_DXT3, s2.DXT5: s2.GL_DXT5}
DITHERS = ["NONE", "SIMPLE", "FLOYDSTEINBERG"]
REFINES = ["NEVER", "ALWAYS", "LOOP"]
MASK = (1 << 32) - 1


def listed():
    return [
        # a late mip level: the call is all latency
        dict(name="txc_mip_20x12", kind="txc", width=20, height=12, comps=4, gen="sinus", dxt=s2.DXT1, cd=s2.WAVG,
             nrandom=-1, refine=s2.REFINE_ALWAYS, dither=s2.DITHER_SIMPLE),
        # a small texture with the library's default settings (the benchmark's first single-image workload)
        dict(name="txc_sinus_256", kind="txc", width=256, height=256, comps=4, gen="sinus", dxt=s2.DXT1, cd=s2.WAVG,
             nrandom=-1, refine=s2.REFINE_ALWAYS, dither=s2.DITHER_SIMPLE),
        # a large texture with alpha at high quality (the benchmark's second single-image workload)
        dict(name="txc_tiles_4096", kind="txc", width=4096, height=4096, comps=4, gen="tiles", dxt=s2.DXT5,
             cd=s2.SRGB_MIXED, nrandom=0, refine=s2.REFINE_LOOP, dither=s2.DITHER_SIMPLE),
        # an asset build with the CLI's best-quality setting: Floyd-Steinberg, 32 random colours
        dict(name="txc_fs_rand32_1024", kind="txc", width=1024, height=1024, comps=4, gen="sinus", dxt=s2.DXT1,
             cd=s2.SRGB_MIXED, nrandom=32, refine=s2.REFINE_LOOP, dither=s2.DITHER_FLOYDSTEINBERG),
        # a frame-sized atlas encoded on the device in quick mode
        dict(name="quick_wavg_dxt1_16384", kind="encode", width=16384, height=16384, gen="sinus", raw=True,
             dxt=s2.DXT1, cd=s2.WAVG, nrandom=-1, refine=s2.REFINE_ALWAYS),
        # quick mode with an expensive distance on a size that no tile divides
        dict(name="quick_srgb_dxt5_4093x2047", kind="encode", width=4093, height=2047, gen="tiles", raw=True,
             dxt=s2.DXT5, cd=s2.SRGB, nrandom=-1, refine=s2.REFINE_LOOP),
        # a normal map at best quality from quantized texels
        dict(name="rand64_normalmap_4096", kind="encode", width=4096, height=4096, gen="normal", raw=False,
             dxt=s2.DXT1, cd=s2.NORMALMAP, nrandom=64, refine=s2.REFINE_LOOP),
        # an asset set: textures of all sizes, formats and distances with their mip chains
        dict(name="batch_200_textures", kind="batch", count=200, spec_seed=workloads.BATCH_SEED, serve_mix=False),
        # a large encoded texture read back
        dict(name="decode_dxt5_8192", kind="decode", width=8192, height=8192, dxt=s2.DXT5),
        # the quality of an encoding
        dict(name="error_wavg_2048", kind="error", width=2048, height=2048, gen="sinus", raw=True, dxt=s2.DXT1,
             cd=s2.WAVG),
        # the mip chain of an uploaded texture
        dict(name="mip_chain_4096", kind="mip", width=4096, height=4096),
        # a DXT5 texture of 8192 x 8192 made patent-free
        dict(name="s3tc_dxt5_4m_blocks", kind="s3tc", nblocks=1 << 22, dxt=s2.DXT5),
    ]


def _size(rng, lo, hi, odd=0.5):
    """A side length spread over the logarithm of [lo, hi]; about half of them are powers of two."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() >= odd:
        v = 1 << int(round(math.log2(v)))
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["txc", "txc", "encode", "encode", "batch", "decode", "error", "mip", "s3tc"])
    dxt = rng.choice([s2.DXT1, s2.DXT3, s2.DXT5])
    if kind == "batch":
        return dict(kind=kind, count=rng.randint(8, 120), spec_seed=rng.randint(100, 1 << 20),
                    serve_mix=rng.random() < 0.3)
    if kind == "s3tc":
        return dict(kind=kind, nblocks=_size(rng, 1, 1 << 22, 0.8), dxt=dxt)
    if kind == "mip":
        return dict(kind=kind, width=_size(rng, 2, 4096), height=_size(rng, 2, 4096))
    if kind == "decode":
        return dict(kind=kind, width=_size(rng, 1, 8192), height=_size(rng, 1, 8192), dxt=dxt)
    quality = rng.choice(["quick", "quick", "all16", "random"])
    refine = rng.choice([s2.REFINE_NEVER, s2.REFINE_ALWAYS, s2.REFINE_LOOP])
    cd = rng.choice([c for c in range(8) if quality != "quick" or c != s2.NORMALMAP])
    gen = "normal" if cd == s2.NORMALMAP else rng.choice(["sinus", "tiles"])
    if kind == "error":
        return dict(kind=kind, width=_size(rng, 4, 2048), height=_size(rng, 4, 2048), gen=gen, raw=True, dxt=dxt, cd=cd)
    nrandom = {"quick": -1, "all16": 0, "random": rng.choice([8, 32, 64])}[quality]
    if kind == "txc":
        dither = rng.choice([s2.DITHER_NONE, s2.DITHER_SIMPLE, s2.DITHER_SIMPLE, s2.DITHER_FLOYDSTEINBERG])
        hi = 1024 if quality == "random" or dither == s2.DITHER_FLOYDSTEINBERG else 4096
        return dict(kind=kind, width=_size(rng, 4, hi), height=_size(rng, 4, hi), comps=rng.choice([3, 4, 4]), gen=gen,
                    dxt=dxt, cd=cd, nrandom=nrandom, refine=refine, dither=dither)
    hi = {"quick": 8192, "all16": 2048, "random": 1024}[quality]
    return dict(kind=kind, width=_size(rng, 4, hi), height=_size(rng, 4, hi), gen=gen, raw=rng.random() < 0.7, dxt=dxt,
                cd=cd, nrandom=nrandom, refine=refine)


# ---- inputs ----

def _image(gen, width, height, seed):
    """height x width x 4 uint8 on the GPU: what textures look like."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    noise = lambda *shape: torch.rand(*shape, device="cuda", generator=g)
    par = noise(64).tolist()
    x = torch.arange(width, device="cuda", dtype=torch.float32)
    y = torch.arange(height, device="cuda", dtype=torch.float32)[:, None]
    out = torch.empty(height, width, 4, dtype=torch.uint8, device="cuda")
    if gen == "normal":  # the normals of a height field of waves
        gx = torch.zeros(height, width, device="cuda")
        gy = torch.zeros(height, width, device="cuda")
        for k in range(6):
            fx, fy = 0.002 + 0.05 * par[4 * k], 0.002 + 0.05 * par[4 * k + 1]
            c = torch.cos(x * fx + y * fy + 6.28 * par[4 * k + 2]) * (0.05 + 0.2 * par[4 * k + 3])
            gx -= c
            gy += c * (0.3 + par[24 + k])
        inv = torch.rsqrt(gx * gx + gy * gy + 1)
        for ch, n in enumerate((gx * inv, gy * inv, inv)):
            out[..., ch] = (n * 127.5 + 128).clamp_(0, 255)
        out[..., 3] = 255
        return out
    for ch in range(3):
        if gen == "sinus":  # smooth colours with a little noise
            f = torch.sin(x * (0.01 + 0.05 * par[4 * ch]) + 6 * par[4 * ch + 1]) * torch.sin(
                y * (0.01 + 0.05 * par[4 * ch + 2]) + 6 * par[4 * ch + 3])
            v = f.mul_(110).add_(128)
            v.add_(noise(height, width).mul_(16).sub_(8))
        else:  # tiles of flat gradients with hard edges
            tx, ty = torch.floor(x / 64), torch.floor(y / 64)
            base = torch.frac(torch.abs(torch.sin(tx * 12.9898 + ty * 78.233 + ch * 37.7 + par[40 + ch])) * 43758.5)
            v = base.mul_(160).add_((x % 64) * (0.3 + par[44 + ch])).add_((y % 64) * (0.3 + par[48 + ch]))
        out[..., ch] = v.clamp_(0, 255)
        del v
    if gen == "sinus":
        out[..., 3] = 255
    else:  # an alpha ramp from the middle, with speckles
        r = torch.sqrt((x - width / 2) ** 2 + (y - height / 2) ** 2)
        a = 255 - r * (255 / (0.5 * max(width, height)))
        out[..., 3] = torch.where(noise(height, width) < 0.02, 255 - a, a).clamp_(0, 255)
    return out


def _quantized(img, dxt):
    """What rgb565_image leaves with DITHER_NONE."""
    a = {s2.DXT1: 7, s2.DXT3: 4, s2.DXT5: 0}[dxt]
    shift = torch.tensor([3, 2, 3, a], dtype=torch.uint8, device="cuda")
    return torch.bitwise_right_shift(img, shift)


def _random_bytes(n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randint(0, 256, (n,), dtype=torch.uint8, device="cuda", generator=g)


def _device_blocks(img, raw, c, nrandom=-1):
    h, w = img.shape[:2]
    out = torch.zeros(s2.nblocks(w, h) * s2.block_bytes(c["dxt"]), dtype=torch.uint8, device="cuda")
    s2.encode_image_device(img.data_ptr(), s2.SRC_RGBA8 if raw else s2.SRC_QUANTIZED, w, h, out.data_ptr(), c["dxt"],
                           c.get("cd", s2.WAVG), nrandom, s2.REFINE_ALWAYS)
    return out


def _specs(c):
    return synth.batch_specs(c["count"], c["spec_seed"], c["serve_mix"])


def _prepare_batch(c, seed):
    """A set of textures on the device with their mip levels, and the plan that encodes them."""
    specs = _specs(c)
    layouts = [s2.mip_layout(s.width, s.height) for s in specs]
    base, total = [], 0
    for _, size in layouts:
        base.append(total)
        total += size
    host = np.zeros(total, np.uint8)
    for s, b in zip(specs, base):
        s.seed = (s.seed ^ (seed * 0x9E3779B97F4A7C15)) & ((1 << 64) - 1)
        host[b:b + s.width * s.height * 4] = synth.texture(s)
    src = torch.from_numpy(host).cuda()
    torch.cuda.synchronize()
    s2.mip_chain_batch([(src.data_ptr() + b, s.width, s.height) for s, b in zip(specs, base)])
    jobs, out = [], 0
    for s, b, (levels, _) in zip(specs, base, layouts):
        for k, (off, w, h) in enumerate(levels):
            jobs.append((b + off, out, w, h, s.dxt, s.cd, s.nrandom, s.refine, workloads.level_seed(s.seed, k)))
            out += (s2.nblocks(w, h) * s2.block_bytes(s.dxt) + 255) & ~255
    dst = torch.zeros(out, dtype=torch.uint8, device="cuda")
    arr = (s2.Job * len(jobs))(*[s2.Job(src.data_ptr() + i, dst.data_ptr() + o, w, h, s2.SRC_RGBA8, d, cd, nr, rf, sd)
                                 for i, o, w, h, d, cd, nr, rf, sd in jobs])
    batch = s2.Batch(SimpleNamespace(jobs=arr))
    return dict(src=src, dst=dst, batch=batch)


def prepare(case, seed):
    c = case
    seed &= MASK
    st = dict(case=c, seed=seed)
    kind = c["kind"]
    if kind == "batch":
        st.update(_prepare_batch(c, seed))
        return st
    if kind == "s3tc":
        st["src"] = _random_bytes(c["nblocks"] * s2.block_bytes(c["dxt"]), seed)
        st["dst"] = torch.empty_like(st["src"])
        torch.cuda.synchronize()
        return st
    if kind == "mip":
        st["src"] = _image("sinus", c["width"], c["height"], seed)
        st["bytes"] = s2.mip_layout(c["width"], c["height"])[1]
        st["dst"] = torch.zeros(st["bytes"], dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        return st
    if kind == "decode":
        st["src"] = _random_bytes(s2.nblocks(c["width"], c["height"]) * s2.block_bytes(c["dxt"]), seed)
        st["dst"] = torch.empty(c["height"], c["width"], 4, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        return st
    img = _image(c["gen"], c["width"], c["height"], seed)
    nbytes = s2.nblocks(c["width"], c["height"]) * s2.block_bytes(c["dxt"])
    if kind == "txc":
        st["src"] = img[..., :c["comps"]].contiguous().cpu().numpy()
        st["dst"] = np.zeros(nbytes, np.uint8)
        st["env"] = dict(S2TC_DITHER_MODE=DITHERS[c["dither"]], S2TC_COLORDIST_MODE=s2.COLORDIST_NAMES[c["cd"]],
                         S2TC_RANDOM_COLORS=str(c["nrandom"]), S2TC_REFINE_COLORS=REFINES[c["refine"]],
                         S2TC_RANDOM_SEED=str(seed))
        lib = s2.lib()
        lib.tx_compress_dxtn.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p, ctypes.c_uint,
                                         ctypes.c_void_p, ctypes.c_int]
        st["call"] = lib.tx_compress_dxtn
        return st
    st["src"] = img if c["raw"] else _quantized(img, c["dxt"])
    if kind == "error":
        st["blocks"] = _device_blocks(st["src"], c["raw"], c)
    else:
        st["dst"] = torch.zeros(nbytes, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    return st


def run(state):
    c = state["case"]
    kind = c["kind"]
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "txc":
        env = state["env"]
        for k, v in env.items():
            if os.environ.get(k) != v:
                os.environ[k] = v
        w = c["width"]
        state["call"](c["comps"], w, c["height"], state["src"].ctypes.data, GL_FORMATS[c["dxt"]],
                      state["dst"].ctypes.data, (w + 3) // 4 * s2.block_bytes(c["dxt"]))
        return state["dst"]
    if kind == "encode":
        s2.encode_image_device(state["src"].data_ptr(), s2.SRC_RGBA8 if c["raw"] else s2.SRC_QUANTIZED, c["width"],
                               c["height"], state["dst"].data_ptr(), c["dxt"], c["cd"], c["nrandom"], c["refine"],
                               state["seed"], stream)
    elif kind == "batch":
        state["batch"].launch(stream)
    elif kind == "decode":
        s2.decode_image_device(state["src"].data_ptr(), GL_FORMATS[c["dxt"]], c["width"], c["height"],
                               state["dst"].data_ptr(), stream)
    elif kind == "error":
        return s2.colordist_error_device(state["src"].data_ptr(), s2.SRC_RGBA8 if c["raw"] else s2.SRC_QUANTIZED,
                                         c["width"], c["height"], state["blocks"].data_ptr(), c["dxt"], c["cd"], stream)
    elif kind == "mip":
        s2.mip_chain_device(state["src"].data_ptr(), c["width"], c["height"], state["dst"].data_ptr(), state["bytes"],
                            stream)
    else:
        s2.from_s3tc_device(state["src"].data_ptr(), state["dst"].data_ptr(), c["nblocks"], c["dxt"], stream)
    return state["dst"]


# ---- the work of a pass ----

def _encode_work(w, h, comps, dxt, cd, nrandom):
    """Texels in, blocks out; the minima and sums of the candidate pair search where there is one, else two
    distances of about eight operations a texel."""
    nb = s2.nblocks(w, h)
    m = 16 + max(nrandom, 0)
    pairs = 16 * m * (m - 1) if nrandom >= 0 or cd == s2.NORMALMAP else 0
    return comps * w * h + nb * s2.block_bytes(dxt), 16 * w * h + nb * pairs


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("txc", "encode"):
        b, f = _encode_work(c["width"], c["height"], c.get("comps", 4), c["dxt"], c["cd"], c["nrandom"])
    elif kind == "batch":
        b = f = 0
        for s in _specs(c):
            for _, w, h in s2.mip_layout(s.width, s.height)[0]:
                jb, jf = _encode_work(w, h, 4, s.dxt, s.cd, s.nrandom)
                b, f = b + jb, f + jf
    elif kind == "s3tc":
        b, f = 2 * c["nblocks"] * s2.block_bytes(c["dxt"]), 0
    elif kind == "mip":
        b = 4 * c["width"] * c["height"] + sum(4 * w * h for _, w, h in s2.mip_layout(c["width"], c["height"])[0])
        f = 0
    else:  # decode, error
        n = c["width"] * c["height"]
        b = 4 * n + s2.nblocks(c["width"], c["height"]) * s2.block_bytes(c["dxt"])
        f = 8 * n if kind == "error" else 0
    return {"bytes": b, "flops": f}


def exact(case, seed):
    """Every output is an encoding, decoded bytes or a whole number: none is rounded."""
    return None
