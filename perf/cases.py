"""The work this framework is used for, as cases that can be timed: frames coded one at a time,
batches of frames, frames of a served stream, and frames decoded, each through the entry points
a program calls.

Inputs are the seeded synthetic frames of the repository's benchmark (smooth waves, rectangles,
noise of sigma 30) at the DCI containers and at generic sizes. Outputs are whole: every array of
a frame's Tier-1 result (block records, pass lengths, pass distortions, codeword bytes), whole
codestreams, whole pictures, in buffers of the program's own that are zero past what was
written. They are bytes and whole numbers that must not change, so the tolerance is "exact"
throughout and there is no 64-bit value to compare with."""
import ctypes as C
import math

import numpy as np
import torch

import libgail_amd as g

# An early-termination threshold as a running stream has it: about a quarter of the slope that
# rate control settles on for a 4K frame at 24 frames/s and 250 Mbit/s.
STREAM_SLOPE = 1500.0
FPS, MBPS = 24.0, 250.0

_device = None


def _dev():
    global _device
    if _device is None:
        _device = g.Device(0)
    return _device


# ---------------------------------------------------------------- the cases
def _frame(name, w, h, fourk, fmt="xyz", slope=0.0, rate=False):
    return {"name": name, "kind": "frame", "w": w, "h": h, "fourk": fourk, "fmt": fmt, "slope": slope, "rate": rate}


def _batch(name, frames, slope=0.0, rate=False, graph=False):
    """frames: "count x container or WxH x format" groups joined by ','."""
    return {"name": name, "kind": "batch", "frames": frames, "slope": slope, "rate": rate, "graph": graph}


def _decode(name, w, h, fourk, reduce=0, high_bits=True, hbm=False):
    return {"name": name, "kind": "decode", "w": w, "h": h, "fourk": fourk, "reduce": reduce, "high_bits": high_bits,
            "hbm": hbm}


def listed():
    return [
        # a tile or proxy frame coded alone: launches and latency are all of it
        _frame("frame_512x256", 512, 256, 0),
        # an odd-sized picture, every block row and column ragged
        _frame("frame_1357x771", 1357, 771, 0),
        # the plain encoder, one frame per call, in a running 2K stream (rate control is left to
        # the host) and a 4K stream (rate control on the device, as the library API runs it)
        _frame("frame_2k_flat", 1998, 1080, 0, slope=STREAM_SLOPE),
        _frame("frame_4k_flat_rate", 3996, 2160, 1, slope=STREAM_SLOPE, rate=True),
        # HDR R'G'B' with tone mapping, all passes kept (a stream's first frame has no threshold)
        _frame("frame_4k_scope_hdr", 4096, 1716, 1, fmt="rgb48"),
        # the batched form: 12 2K frames resident in HBM, the whole Tier-1 output to the host
        _batch("batch_12_2k_flat", "12x2k_flatxxyz", slope=STREAM_SLOPE),
        # a served job: 16 4K frames with rate control on the device
        _batch("batch_16_4k_flat_rate", "16x4k_flatxxyz", slope=STREAM_SLOPE, rate=True),
        # a mixed job: sizes and input formats, no early termination, replayed as a graph
        _batch("batch_mixed_8", "2x2k_flatxgbrp12,2x2k_scopexxyz,2x4k_scopexyuv420p10,2x4k_fullxxyz", rate=True,
               graph=True),
        # the decoder on host buffers at 2K; on buffers in HBM at 4K; a 4K frame at half size
        _decode("decode_2k_flat", 1998, 1080, 0),
        _decode("decode_4k_flat", 3996, 2160, 1, hbm=True),
        _decode("decode_4k_half", 3996, 2160, 1, reduce=1, high_bits=False, hbm=True),
        # the served form: a closed burst of 4K frames to codestreams
        {"name": "served_32_4k_flat", "kind": "served", "count": 32, "container": "4k_flat", "slope": STREAM_SLOPE},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng):
    w, h = _log(rng, 128, 4096), _log(rng, 128, 2160)
    return w, h, 1 if w > 2048 or h > 1080 else rng.randrange(2)


def draw(rng):
    kind = rng.choice(["frame", "frame", "batch", "batch", "decode", "decode", "served"])
    if kind == "frame":
        w, h, k = _size(rng)
        c = _frame("", w, h, k, rng.choice(["xyz", "xyz", "rgb48", "yuv420p10", "gbrp12"]),
                   rng.choice([0.0, 300.0, STREAM_SLOPE]), rng.random() < 0.5)
    elif kind == "batch":
        groups, pixels = [], 0
        for _ in range(rng.randint(1, 3)):
            n = _log(rng, 1, 5)
            if rng.random() < 0.6:
                size = rng.choice(sorted(g.CONTAINERS))
                w, h, _ = g.CONTAINERS[size]
            else:
                w, h, _ = _size(rng)
                size = "%dx%d" % (w, h)
            n = max(1, min(n, (12 * 3996 * 2160 - pixels) // (w * h)))
            pixels += n * w * h
            groups.append("%dx%sx%s" % (n, size, rng.choice(["xyz", "xyz", "yuv420p10", "gbrp12"])))
        c = _batch("", ",".join(groups), rng.choice([0.0, STREAM_SLOPE]), rng.random() < 0.5, rng.random() < 0.3)
    elif kind == "decode":
        w, h, k = _size(rng)
        c = _decode("", w, h, k, rng.choice([0, 0, 0, 1, 2]), rng.random() < 0.5, rng.random() < 0.5)
    else:
        c = {"name": "", "kind": "served", "count": rng.randint(3, 24), "container": rng.choice(sorted(g.CONTAINERS)),
             "slope": rng.choice([300.0, STREAM_SLOPE])}
    del c["name"]
    return c


def _groups(case):
    """(width, height, 4K decomposition, format) of every frame of a batch case."""
    out = []
    for group in case["frames"].split(","):
        n, rest = group.split("x", 1)
        size, fmt = next((rest[:-len(f) - 1], f) for f in ("xyz", "yuv420p10", "gbrp12", "rgb48")
                         if rest.endswith("x" + f))
        if size in g.CONTAINERS:
            w, h, k = g.CONTAINERS[size]
        else:
            w, h = (int(v) for v in size.split("x"))
            k = 1 if w > 2048 or h > 1080 else 0
        out += [(w, h, k, fmt)] * int(n)
    return out


# ---------------------------------------------------------------- inputs
def _picture(seed, w, h, fmt):
    """A frame in the encoder's input layout, derived from a synthetic frame."""
    x = g.synth_frame(seed, w, h, threads=16)
    if fmt == "xyz":
        return x
    if fmt == "rgb48":
        return np.ascontiguousarray((x << 4).transpose(1, 2, 0))
    if fmt == "gbrp12":
        return np.concatenate([x[1].ravel(), x[2].ravel(), x[0].ravel()])
    return np.concatenate([(x[1] >> 2).ravel(), (x[0, ::2, ::2] >> 2).ravel(), (x[2, ::2, ::2] >> 2).ravel()])


def _settings(layout, fmt):
    if fmt == "xyz":
        return g.xyz_settings(layout)
    if fmt == "rgb48":  # PQ, BT.2020, the shoulder tone map
        return g.rgb48_settings(layout, transfer=2, primaries=1, tone_map=1)
    if fmt == "gbrp12":
        return g.planar_settings(layout, 12, 0, 0, 1, 1)
    return g.planar_settings(layout, 10, 1, 1, 0, 0)


def _pinned(a):
    """The frame in pinned host memory, which a program that streams frames reads them into."""
    p = g.pinned_empty(a.nbytes).view(a.dtype).reshape(a.shape)
    p[...] = a
    return p


class _State:
    """What a program holds; the plugin's objects close with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for o in self.__dict__.pop("objects", []):
            o.close()


class _Keep:
    """Where a program keeps one frame's Tier-1 result, which the encoder's own buffers hold only
    until its next frame."""

    def __init__(self, layout, rate):
        n, px = layout.num_cblks, layout.width * layout.height
        nbytes = min(3 * px + 65536, int(MBPS * 1e6 / 8 / FPS) + 4 * n) if rate else 3 * px + 65536
        self.arrays = [torch.zeros(5 * n, dtype=torch.int32), torch.zeros(40 * n, dtype=torch.int32),
                       torch.zeros(40 * n, dtype=torch.int32), torch.zeros(nbytes, dtype=torch.uint8)]

    def take(self, t1):
        r = g.Tier1Result(t1, copy=False)
        for dst, src in zip(self.arrays, (r.info.reshape(-1).view(np.int32), r.pass_len.view(np.int32), r.pass_dist,
                                          r.data)):
            dst[:len(src)].copy_(torch.from_numpy(src))
        return self.arrays


def _distinct(seed, frames):
    """Inputs of a batch: up to two distinct synthetic frames per geometry and format, the rest
    the same frames rolled by some rows (other blocks, other symbols)."""
    made, out = {}, []
    for i, (w, h, _, fmt) in enumerate(frames):
        have = made.setdefault((w, h, fmt), [])
        k = len(have)
        if k < 2:
            have.append(_picture(1000 * seed + i, w, h, fmt))
            out.append(have[k])
        else:
            have.append(None)
            out.append(np.roll(have[k % 2].reshape(-1), 1 + 2 * w * (17 * k)).reshape(have[0].shape))
    return out


def prepare(case, seed):
    dev = _dev()
    kind = case["kind"]
    if kind == "frame":
        layout = g.FrameLayout(case["w"], case["h"], case["fourk"])
        settings = _settings(layout, case["fmt"])
        if case["rate"]:
            settings = g.with_rate_control(settings, FPS, MBPS)
        enc = g.Encoder(dev, layout, settings)
        enc.set_slope(case["slope"])
        return _State(kind=kind, enc=enc, frame=_pinned(_picture(seed, case["w"], case["h"], case["fmt"])),
                      keep=_Keep(layout, case["rate"]), objects=[enc])
    if kind == "batch":
        frames = _groups(case)
        layouts = [g.FrameLayout(w, h, k) for w, h, k, _ in frames]
        settings = [_settings(L, f[3]) for L, f in zip(layouts, frames)]
        if case["rate"]:
            settings = [g.with_rate_control(s, FPS, MBPS) for s in settings]
        b = g.Batch(dev, layouts, settings, use_graph=case["graph"])
        for i, x in enumerate(_distinct(seed, frames)):
            b.upload(i, x)
            b.set_slope(i, case["slope"])
        return _State(kind=kind, batch=b, keep=[_Keep(L, case["rate"]) for L in layouts], objects=[b])
    if kind == "decode":
        # a frame coded at the DCI rate: the passes that rate control keeps
        w, h, k = case["w"], case["h"], case["fourk"]
        layout = g.FrameLayout(w, h, k)
        b = g.Batch(dev, [layout], [g.with_rate_control(g.xyz_settings(layout), FPS, MBPS)])
        b.upload(0, g.synth_frame(seed, w, h, threads=16))
        b.set_slope(0, STREAM_SLOPE)
        (t1,), _ = b.encode()
        b.close()
        blocks = g.block_table(t1)
        dec = g.Decoder(dev, layout, case["reduce"], case["high_bits"])
        ow, oh = g.decoded_size(layout, case["reduce"])
        if case["hbm"]:
            data = torch.from_numpy(t1.data).cuda()
            out = torch.zeros((oh, 3 * ow), dtype=torch.int16, device="cuda")
            torch.cuda.synchronize()
            src, dst = (data.data_ptr(), data.numel()), (out.data_ptr(), 6 * ow)
        else:
            data = src = _pinned(t1.data)
            out = dst = g.pinned_empty(6 * ow * oh).view(np.uint16).reshape(oh, 3 * ow)
        return _State(kind=kind, dec=dec, data=data, src=src, blocks=blocks, out=out, dst=dst, objects=[dec])
    # served: frames resident in HBM, every job made and run once before the stream
    w, h, _ = g.CONTAINERS[case["container"]]
    planes = [g.DeviceFrame(list(g.synth_frame(100 * seed + i, w, h, threads=16))) for i in range(2)]
    cfg = g.stream_config(case["container"], "xyz12_planar", fps=FPS, mbps=MBPS)
    srv = g.Server(check=True, keep=True)
    s = _State(kind=kind, srv=srv, cfg=cfg, planes=planes, count=case["count"], slope=case["slope"], next_id=0,
               out=[torch.zeros(int(MBPS * 1e6 / 8 / FPS), dtype=torch.uint8) for _ in range(case["count"])],
               objects=[srv] + planes)
    run(s)
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    s = state
    if s.kind == "frame":
        out, tm = g.Tier1(), g.FrameTimings()
        g._check(g.plugin().encoder_encode(s.enc.handle, s.frame.ctypes.data, C.byref(out), C.byref(tm), None), "encode")
        return s.keep.take(out)
    if s.kind == "batch":
        b = s.batch
        b.launch()
        outs, tm = (g.Tier1 * b.n)(), g.FrameTimings()
        g._check(g.plugin().batch_wait(b.handle, outs, C.byref(tm)), "batch_wait")
        return [k.take(t) for k, t in zip(s.keep, outs)]
    if s.kind == "decode":
        s.dec.decode(s.src, s.blocks, out=s.dst)
        return s.out
    ids = range(s.next_id, s.next_id + s.count)
    s.next_id += s.count
    for i in ids:
        s.srv.submit(i, 1, s.cfg, s.planes[i % len(s.planes)], s.slope)
    s.srv.drain()
    results = [s.srv.results.pop(i) for i in ids]
    for r, out in zip(results, s.out):
        if r["status"] != 0:
            raise RuntimeError("a served frame failed")
        out[:r["size"]].copy_(torch.frombuffer(bytearray(r["codestream"]), dtype=torch.uint8))
    return s.out


# ---------------------------------------------------------------- work and tolerance
def work(case):
    """Bytes: each frame read once and its coded form (or picture) written once. Operations per
    sample: about 40 for the transform (9/7 lifting in both directions over all levels, DC shift,
    component transform) and 10 for each of the arithmetic coder's symbols, about 3.6 a sample in
    coding (measured on these frames, early termination on) and 0.6 in decoding at the DCI rate."""
    kind = case["kind"]
    rate_bytes = MBPS * 1e6 / 8 / FPS
    if kind == "frame":
        frames, rate = [(case["w"], case["h"], case["fourk"], case["fmt"])], case["rate"]
    elif kind == "batch":
        frames, rate = _groups(case), case["rate"]
    elif kind == "served":
        frames, rate = [g.CONTAINERS[case["container"]] + ("xyz",)] * case["count"], True
    else:
        n = 3 * case["w"] * case["h"] / 4 ** case["reduce"]
        code = min(rate_bytes, case["w"] * case["h"] * 1.3)
        return {"bytes": code + 2 * n, "flops": 46 * n}
    nbytes = flops = 0
    for w, h, _, fmt in frames:
        px = w * h
        nbytes += px * (3 if fmt == "yuv420p10" else 6) + (min(rate_bytes, 1.3 * px) if rate else 1.3 * px)
        flops += 3 * px * 76
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    return "exact"
