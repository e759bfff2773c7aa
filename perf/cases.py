"""Performance cases: what programs have this library do, through its public entry points.

Kinds of program:
  frame     An emulator with device-resident RDRAM: hand over one frame's command words, write the VI
            registers, scan out (scanout_sync); the picture is the result.  With `upscale` (and
            `super_sample`) the processor renders and scans out at 2, 4 or 8 times the resolution.
  coherent  An emulator whose own memory is RDRAM: hand over one frame's command words, idle; RDRAM as
            the caller then sees it (colour, depth and everything else in it) is the result.
  scanout   The VI alone: a finished frame shown again, interlaced and blended with the previous
            field, as the conformance driver of the reference scans out (blend_previous_frame on,
            upscale_deinterlacing off).
  batch     Many instances rendered together from fresh command words: enqueue every instance's
            frame, one batch_flush, an asynchronous scanout of each; the pictures are the result.
  recorded  Many instances whose commands are recorded once and replayed from device memory as one
            graph (several frames each), then an asynchronous scanout of each.

Render modes are the three workloads of this package: `shaded` (Gouraud + Z), `textured` (RGBA16
texture, perspective, bilinear, alpha blend, RGBA8888) and `two_cycle` (CI4/CI8 with TLUT, mip LOD, fog,
coverage AA, a fifth texture rectangles).  `mixed` gives each instance one of them with its own size and
primitive count.
"""
import importlib
import math
import os
import random
import sys

import numpy as np

_PACKAGE = os.path.join(os.getcwd(), "parallel-rdp_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)
rdp_mi = importlib.import_module("rdp_mi")
rs = importlib.import_module("rdp_streams")

VI_TYPE_RGBA8888 = 3
VI_SERRATE = 1 << 6
MODES = ("shaded", "textured", "two_cycle")


def listed():
    return [
        # The smallest call: a menu or loading screen, 32 triangles, in the caller's own RDRAM.
        dict(name="coherent_shaded_32", kind="coherent", mode="shaded", width=320, height=240, prims=32),
        # An ordinary 240-line frame of untextured geometry (256 full-screen triangles).
        dict(name="frame_shaded_256", kind="frame", mode="shaded", width=320, height=240, prims=256, upscale=1,
             super_sample=False),
        # A busy high-resolution frame at 32 bits: 4096 textured triangles of 2-200 pixels.
        dict(name="frame_textured_4096", kind="frame", mode="textured", width=640, height=480, prims=4096, upscale=1,
             super_sample=False),
        # The heaviest pixel pipeline at high resolution, with the VI's AA, divot and dither filters.
        dict(name="frame_two_cycle_2560", kind="frame", mode="two_cycle", width=640, height=480, prims=2560, upscale=1,
             super_sample=False),
        # A game frame of odd size in the caller's own RDRAM.
        dict(name="coherent_two_cycle_700", kind="coherent", mode="two_cycle", width=357, height=239, prims=700),
        # The caller's own RDRAM, high resolution, 32 bits.
        dict(name="coherent_textured_1500", kind="coherent", mode="textured", width=640, height=480, prims=1500),
        # A paused or repeated frame: the VI only.
        dict(name="scanout_interlaced", kind="scanout", mode="two_cycle", width=640, height=480, prims=512),
        # Upscaled emulation: 2x of a 240-line textured frame.
        dict(name="upscaled_2x_textured", kind="frame", mode="textured", width=320, height=240, prims=1024, upscale=2,
             super_sample=False),
        # 4x of a high-resolution two-cycle frame.
        dict(name="upscaled_4x_two_cycle", kind="frame", mode="two_cycle", width=640, height=480, prims=2560, upscale=4,
             super_sample=False),
        # 16 instances from fresh commands, one submission.
        dict(name="batch_16_mixed", kind="batch", mode="mixed", instances=16, frames=1, upscale=1, super_sample=False),
        # 16 instances, super-sampled readback with dither at 2x, replayed as one graph.
        dict(name="recorded_16_super_sampled", kind="recorded", mode="mixed", instances=16, frames=2, upscale=2,
             super_sample=True),
        # Many instances and frames replayed as one graph: the throughput form.
        dict(name="recorded_32x8_mixed", kind="recorded", mode="mixed", instances=32, frames=8, upscale=1,
             super_sample=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_MOST_PRIMS = {"shaded": 512, "textured": 4096, "two_cycle": 2560}


def draw(rng):
    kind = rng.choice(("coherent", "frame", "frame", "scanout", "upscaled", "batch", "recorded"))
    if kind in ("batch", "recorded"):
        upscale = rng.choice((1, 1, 2)) if kind == "recorded" else 1
        frames = 1 if kind == "batch" else rng.randint(1, 8 if upscale == 1 else 2)
        return dict(kind=kind, mode="mixed", instances=_log_int(rng, 2, 32 if upscale == 1 else 16), frames=frames,
                    upscale=upscale, super_sample=upscale > 1 and rng.random() < 0.5)
    mode = rng.choice(MODES)
    # Widths from 256 up: the range every front end of the reference uses, and what upscaling needs.
    case = dict(kind=kind, mode=mode, width=rng.randint(256, 640), height=rng.randint(200, 480),
                prims=_log_int(rng, 16, _MOST_PRIMS[mode]))
    if kind == "upscaled":
        case.update(kind="frame", upscale=rng.choice((2, 2, 4, 4, 8)), super_sample=rng.random() < 0.3)
        if case["upscale"] == 8:
            case.update(width=rng.randint(256, 320), height=rng.randint(200, 240), prims=_log_int(rng, 16, 512))
    elif kind == "frame":
        case.update(upscale=1, super_sample=False)
    return case


def _stream(mode, width, height, prims, frames, seed):
    """(initial RDRAM words, command words of every frame, bytes per pixel) of one seeded workload."""
    if mode == "shaded":
        streams = [rs.config0_stream(seed=seed + 7919 * f, num_triangles=prims, width=width, height=height)
                   for f in range(frames)]
        return np.zeros(rs.RDRAM_SIZE // 4, np.uint32), [s.frames[0].words for s in streams], 2
    make = rs.config1_stream if mode == "textured" else rs.config2_stream
    s = make(seed, frames, prims, width, height)
    return s.rdram_init, [f.words for f in s.frames], 4 if mode == "textured" else 2


def _vi_registers(width, height, pixel_bytes, interlaced=False):
    regs = dict(rs.c2_vi_registers(width, height))
    if pixel_bytes == 4:
        regs[rs.VI_CONTROL] = (regs[rs.VI_CONTROL] & ~3) | VI_TYPE_RGBA8888
    if interlaced:
        regs[rs.VI_CONTROL] |= VI_SERRATE
    return regs


def _flags(case):
    flags = rdp_mi.FLAG_UPSCALING.get(case.get("upscale", 1), 0)
    if case.get("super_sample"):
        flags |= rdp_mi.FLAG_SUPER_SAMPLED_READ_BACK | rdp_mi.FLAG_SUPER_SAMPLED_DITHER
    return flags


def _processor(case, rdram):
    p = rdp_mi.CommandProcessor(rs.RDRAM_SIZE, flags=_flags(case))
    p.write_rdram(rdram)
    p.write_hidden_rdram(np.zeros(rs.RDRAM_SIZE // 2, np.uint8))
    return p


def _set_registers(p, regs):
    for reg, value in regs.items():
        p.set_vi_register(reg, value)


def _instance(rng, i):
    """Mode, size and primitive count of one instance of a mixed batch."""
    mode = MODES[i % 3]
    width, height = rng.choice(((320, 240), (320, 240), (640, 480), (rng.randint(256, 640), rng.randint(200, 480))))
    return mode, width, height, _log_int(rng, 32, _MOST_PRIMS[mode])


def prepare(case, seed):
    kind = case["kind"]
    seed = int(seed) & 0x3FFFFFFF
    if kind in ("batch", "recorded"):
        rng = random.Random(seed)
        # Sizes belong to the case and contents to the seed: two seeds cost the same.
        sizes = random.Random(1000 * case["instances"] + case["frames"])
        procs, words, buffers = [], [], []
        for i in range(case["instances"]):
            mode, width, height, prims = _instance(sizes, i)
            rdram, frames, pixel_bytes = _stream(mode, width, height, prims, case["frames"], rng.getrandbits(30))
            p = _processor(case, rdram)
            p.hold_submissions()
            _set_registers(p, _vi_registers(width, height, pixel_bytes))
            procs.append(p)
            words.append(np.concatenate(frames))
            buffers.append(rdp_mi.ScanoutBuffer())
        state = dict(kind=kind, procs=procs, words=words, buffers=buffers)
        if kind == "recorded":
            for p, w in zip(procs, words):
                p.enqueue_commands(w)
            state["recording"] = rdp_mi.Recording(procs, batched=True)
        return state

    rdram, frames, pixel_bytes = _stream(case["mode"], case["width"], case["height"], case["prims"], 1, seed)
    if kind == "coherent":
        memory = np.array(rdram)
        p = rdp_mi.CommandProcessor(rs.RDRAM_SIZE, host_rdram=memory)
        p.write_hidden_rdram(np.zeros(rs.RDRAM_SIZE // 2, np.uint8))
        return dict(kind=kind, proc=p, words=frames[0], memory=memory)
    p = _processor(case, rdram)
    regs = _vi_registers(case["width"], case["height"], pixel_bytes, interlaced=kind == "scanout")
    state = dict(kind=kind, proc=p, words=frames[0], regs=regs)
    if kind == "scanout":
        p.enqueue_commands(frames[0])
        _set_registers(p, regs)
        p.idle()
        state["options"] = rdp_mi.ScanoutOptions.default(blend_previous_frame=1, upscale_deinterlacing=0)
    return state


def run(state):
    kind = state["kind"]
    if kind == "frame":
        p = state["proc"]
        p.enqueue_commands(state["words"])
        _set_registers(p, state["regs"])
        return p.scanout_sync().view(np.int32)
    if kind == "coherent":
        p = state["proc"]
        p.enqueue_commands(state["words"])
        p.idle()
        return state["memory"].view(np.int32)
    if kind == "scanout":
        return state["proc"].scanout_sync(state["options"]).view(np.int32)
    procs, buffers = state["procs"], state["buffers"]
    if kind == "batch":
        for p, words in zip(procs, state["words"]):
            p.enqueue_commands(words)
        rdp_mi.batch_flush(procs)
    else:
        state["recording"].replay(1, use_graph=True)
    for p, b in zip(procs, buffers):
        p.scanout_async(b)
    return [b.wait().view(np.int32) for b in buffers]


# Command words of one primitive (a fifth of the two-cycle ones are rectangles of 4 words).
_WORDS = {"shaded": 28, "textured": 44, "two_cycle": 36}
_TEXTURES = {"shaded": 0, "textured": 8 * 2048, "two_cycle": 8 * 8192}


def work(case):
    """Bytes of one pass: the command words and textures read once, colour, depth and their hidden bits
    written once per frame (per sample when upscaled), the picture (or the caller's view of the written
    pages) written once.  The operations are 32-bit integer ones and are not counted as flops."""
    samples = case.get("upscale", 1) ** 2
    picture = 640 * 240 * 4 * samples

    def one(mode, width, height, prims, frames):
        pixel = 6 if mode == "textured" else 3
        commands = prims * _WORDS[mode] * 4
        return frames * (commands + width * height * (pixel + 3) * samples) + _TEXTURES[mode]

    if case["kind"] == "scanout":
        return {"bytes": case["width"] * case["height"] * 3 + 640 * 480 * 4, "flops": 0}
    if case["kind"] in ("batch", "recorded"):
        sizes = random.Random(1000 * case["instances"] + case["frames"])
        total = sum(one(*_instance(sizes, i), case["frames"]) for i in range(case["instances"]))
        return {"bytes": total + case["instances"] * picture, "flops": 0}
    total = one(case["mode"], case["width"], case["height"], case["prims"], 1)
    if case["kind"] == "coherent":
        picture = case["width"] * case["height"] * (6 if case["mode"] == "textured" else 4)
    return {"bytes": total + picture, "flops": 0}


def tolerance(case):
    # Every output is whole numbers that the RDP and the VI define bit by bit.
    return "exact"
