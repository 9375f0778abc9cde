"""Workloads of the denoiser, one public call (or one step of a program's loop) a pass.

A case is a plain dict; ``prepare`` makes what a program holds before the call (device-resident
frames, engines, a network), ``run`` makes the call, ``work`` counts what it cannot do without and
``exact`` gives the floating-point results in 64 bits.  Kinds:

  clip    a range of device-resident frames of all planes of a clip (run_device_batch)
  step    one frame of a live clip, in order, all planes (nf3d_run_device_batch, tables made once)
  plugin  one frame through the filter interface that a video plugin binds, from and to host memory
  labels  noise patterns of one plane by regions (training labels, spatially varying denoising)
  dft2d   block DFTs as matrix products, forward and back
  grad    loss and gradients of one training batch of the noise-PSD network
"""
import ctypes
import math

import numpy as np
import torch

import neo_fft3d_amd as nf
from neo_fft3d_amd import learned as nl

DEV = "cuda"

# Defaults of the keys that a clip case does not give (the filter's own defaults, 4:2:0 8-bit video).
CLIP = {"family": "yuv", "ssw": 1, "ssh": 1, "bits": 8, "float": False, "bt": 3, "bw": 32, "bh": 32, "ow": 10, "oh": 10,
        "sigma": 2.0, "sharpen": 0.0, "dehalo": 0.0, "degrid": 1.0, "sigma4": 0.0, "interlaced": 0, "dft": 0, "hidden": 0}


def listed():
    return [
        # One frame of a standard-definition stream at a time with the filter's defaults: the smallest call, its latency.
        {"name": "step_480p_p8", "kind": "step", "width": 640, "height": 480},
        # A plugin's GetFrame: one 1080p frame, host memory to host memory, in order.
        {"name": "plugin_1080p_p8", "kind": "plugin", "width": 1920, "height": 1080, "bw": 48, "bh": 48, "ow": 16, "oh": 16},
        # The benchmark's own workload (1080p 4:2:0, bt=3, 48/16, sharpen), a shot of it.
        {"name": "clip_1080p_p8", "kind": "clip", "width": 1920, "height": 1080, "frames": 64, "bw": 48, "bh": 48, "ow": 16,
         "oh": 16, "sharpen": 0.3},
        # The same with one noise spectrum per block from the network.
        {"name": "learned_1080p_p8", "kind": "clip", "width": 1920, "height": 1080, "frames": 33, "bw": 48, "bh": 48, "ow": 16,
         "oh": 16, "sharpen": 0.3, "hidden": 256},
        # UHD 10-bit with the Kalman mode (recursion over the frames, state in memory).
        {"name": "kalman_2160p_p10", "kind": "clip", "width": 3840, "height": 2160, "frames": 17, "bits": 10, "bt": 0, "sigma": 3.0,
         "ow": 16, "oh": 16},
        # Interlaced standard-definition 4:2:2 10-bit, spatial only: ragged block grid, small planes.
        {"name": "spatial_576i_p10", "kind": "clip", "width": 720, "height": 576, "frames": 25, "ssh": 0, "bits": 10, "bt": 1,
         "interlaced": 1, "sharpen": 0.5},
        # A 4:4:4 16-bit UHD master, the longest temporal window, large blocks, sharpen and dehalo: the largest call.
        {"name": "master_2160p_p16", "kind": "clip", "width": 3840, "height": 2160, "frames": 10, "ssw": 0, "ssh": 0, "bits": 16,
         "bt": 5, "bw": 64, "bh": 64, "ow": 16, "oh": 16, "sharpen": 0.2, "dehalo": 0.5},
        # Float RGB, as in grading: 1283 x 717, no side a multiple of anything.
        {"name": "rgb_float_717p", "kind": "clip", "family": "rgb", "bits": 32, "float": True, "width": 1283, "height": 717,
         "frames": 12, "bw": 48, "bh": 48, "ow": 16, "oh": 16, "sigma": 6.0},
        # The matrix-core precision form of the filter on UHD 10-bit.
        {"name": "precision_2160p_p10", "kind": "clip", "width": 3840, "height": 2160, "frames": 8, "bits": 10, "sigma": 3.0,
         "bw": 48, "bh": 48, "ow": 16, "oh": 16, "dft": 1},
        # The precision form's block transforms alone, the blocks of a UHD plane.
        {"name": "dft2d_32", "kind": "dft2d", "n": 32, "blocks": 32776},
        # Noise labels of a 1080p plane by regions of 4 x 4 blocks.
        {"name": "labels_1080p", "kind": "labels", "width": 1920, "height": 1080, "family": "gray", "bits": 32, "float": True, "bw": 48,
         "bh": 48, "ow": 16, "oh": 16, "rx": 4, "ry": 4},
        # One training batch of the network at the trainer's default size.
        {"name": "grad_4096", "kind": "grad", "d": 1200, "hidden": 256, "batch": 4096},
    ]


def draw(rng):
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["clip"] * 6 + ["step", "plugin", "learned", "labels", "dft2d", "grad"])
    if kind == "grad":
        return {"kind": "grad", "d": rng.choice([16 * 9, 24 * 13 + 4 * 2, 32 * 17, 48 * 25]) // 8 * 8, "hidden": rng.choice([64, 128, 256]),
                "batch": log_int(256, 8192)}
    if kind == "dft2d":
        return {"kind": "dft2d", "n": rng.choice([32, 48, 64]), "blocks": log_int(64, 12000)}
    b = rng.choice([(8, 8), (16, 16), (24, 24), (32, 32), (32, 32), (48, 48), (48, 48), (64, 64), (32, 16), (16, 32)])
    c = {"kind": kind, "bw": b[0], "bh": b[1], "ow": rng.randint(b[0] // 4, b[0] // 2), "oh": rng.randint(b[1] // 4, b[1] // 2)}
    c["width"] = log_int(320, 3840)
    c["height"] = max(240, int(c["width"] * rng.uniform(0.5, 0.8)))
    if kind == "labels":
        c.update(family="gray", bits=32, float=True, rx=rng.randint(1, 8), ry=rng.randint(1, 8))
        return c
    fmt = rng.choice(["yuv420", "yuv420", "yuv422", "yuv444", "gray", "rgb", "rgbs"])
    c["bits"] = rng.choice([8, 8, 10, 16])
    if fmt in ("yuv420", "yuv422"):
        c["width"] -= c["width"] % 2
        c["height"] -= c["height"] % 4
        c["ssh"] = int(fmt == "yuv420")
    elif fmt == "yuv444":
        c.update(ssw=0, ssh=0)
    elif fmt == "gray":
        c["family"] = "gray"
    else:
        c["family"] = "rgb"
        if fmt == "rgbs":
            c.update(bits=32, float=True)
    if kind == "learned":
        c.update(kind="clip", bw=32, bh=32, ow=rng.randint(8, 16), oh=rng.randint(8, 16), hidden=rng.choice([64, 128, 256]))
    c["sigma"] = round(rng.uniform(1.0, 8.0), 2)
    c["bt"] = rng.choice([0, 1, 2, 3, 3, 4, 5]) if c.get("hidden") else rng.choice([-1, 0, 0, 1, 2, 3, 3, 3, 4, 5])
    c["sharpen"] = rng.choice([0.0, 0.0, 0.3, 0.8])
    c["dehalo"] = rng.choice([0.0, 0.0, 0.0, 0.5])
    if c["bt"] == -1 and c["sharpen"] == 0.0 and c["dehalo"] == 0.0:
        c["sharpen"] = 0.5
    c["degrid"] = rng.choice([1.0, 1.0, 0.0])
    if not c.get("hidden") and c["bt"] > -1 and rng.random() < 0.2:
        c["sigma4"] = round(c["sigma"] * 2.5, 2)
    if fmt == "gray" or fmt == "yuv422":
        c["height"] -= c["height"] % 4
        c["interlaced"] = int(rng.random() < 0.3)
    if kind == "clip" and not c.get("hidden") and b in ((32, 32), (48, 48), (64, 64)) and not c.get("float") and rng.random() < 0.2:
        c["dft"] = 1
    if kind in ("clip", "learned"):
        area = c["width"] * c["height"] * (1.0 if fmt == "gray" else 1.5 if fmt == "yuv420" else 2.0 if fmt == "yuv422" else 3.0)
        over = (b[0] / (b[0] - c["ow"])) * (b[1] / (b[1] - c["oh"]))
        c["frames"] = min(max(1, int(60e6 / (area * over) / (3 if c.get("dft") else 1))), log_int(1, 64))
        c["frames"] = max(c["frames"], c["bt"] + 1, 2)
    return c


# ------------------------------------------------------------------ inputs
def full(case):
    return {**CLIP, **case}


def plane_dims(c):
    n = 1 if c["family"] == "gray" else 3
    sub = c["family"] == "yuv"
    return [(c["width"] >> (c["ssw"] if sub and p else 0), c["height"] >> (c["ssh"] if sub and p else 0)) for p in range(n)]


def planes(c, frames, seed):
    """Frames of each plane: a gradient, moving gratings, blocks of texture of different strength, Gaussian noise; in the
    format's samples (16-bit samples as the bits of int16)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    top = 1.0 if c["float"] else float((1 << c["bits"]) - 1)
    out = []
    for p, (w, h) in enumerate(plane_dims(c)):
        y = torch.arange(h, device=DEV, dtype=torch.float32)[:, None]
        x = torch.arange(w, device=DEV, dtype=torch.float32)[None, :]
        r = torch.rand(8, generator=g, device=DEV)
        cell = torch.rand((h // 40 + 1, w // 40 + 1), generator=g, device=DEV).repeat_interleave(40, 0).repeat_interleave(40, 1)[:h, :w]
        fs = []
        for n in range(frames):
            img = 55 + 70 * x / w + 60 * y / h
            img = img + 26 * cell * torch.sin((x * (0.15 + r[0]) + y * r[1] + 1.5 * n) * (0.2 + 0.8 * r[2]) + p)
            img = img + 14 * cell * torch.sin((x * r[3] - y * (0.3 + r[4]) - n) * (0.5 + 2 * r[5]))
            img = img + (3.0 if p == 0 else 2.0) * torch.randn((h, w), generator=g, device=DEV)
            img = (img * (top / 255.0)).clamp(0, top)
            fs.append(img if c["float"] else img.round().to(torch.int32).to(torch.uint8 if c["bits"] == 8 else torch.int16))
        out.append(torch.stack(fs))
    return out


def params(c):
    kw = {k: c[k] for k in ("bt", "bw", "bh", "ow", "oh", "sharpen", "dehalo", "degrid", "interlaced")}
    if c["sigma4"]:
        kw["sigma4"] = c["sigma4"]
    return nf.default_params(c["sigma"], **kw)


def network(d, hidden, batch, level, seed):
    """A network as the trainer sets one up: seeded weights, output bias at the noise level, input normalisation."""
    m = nl.Mlp(d, hidden, d, batch)
    rng = np.random.default_rng(seed)
    m.set_input_norm(level + 1.5 + 0.5 * rng.standard_normal(d), np.full(d, 0.45), 1e-6)
    m.set_params(nl.init_params(d, hidden, d, seed, out_bias=level + 0.2 * rng.standard_normal(d)))
    return m


_stream = None


def stream():
    """The one stream that a program queues its filter calls on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream.cuda_stream


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dft2d":
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        n, nb = case["n"], case["blocks"]
        x = torch.rand((nb, n, n), generator=g, device=DEV) * 1023.0
        return {"case": case, "x": x, "z": torch.empty((nb, n, n // 2 + 1, 2), device=DEV), "y": torch.empty_like(x), "stream": stream()}
    if kind == "grad":
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        d, n, level = case["d"], case["batch"], 9.0
        x = torch.randn((n, d), generator=g, device=DEV).to(torch.bfloat16)
        t = -torch.log(torch.rand((n, d), generator=g, device=DEV).clamp_min(1e-12)) * math.exp(level)
        return {"case": case, "x": x, "t": t, "mlp": network(d, case["hidden"], n, level, seed), "stream": stream()}
    c = full(case)
    if kind == "plugin":
        frames = 24
        host = [p.cpu().numpy() for p in planes(c, frames, seed)]
        fmt = nf.make_format(c["family"], c["bits"], c["float"], c["ssw"], c["ssh"])
        args = "sigma=%g" % c["sigma"] + "".join(";%s=%g" % (k, c[k]) for k in ("bt", "bw", "bh", "ow", "oh", "sharpen", "dehalo", "degrid",
                                                                             "interlaced"))
        if c["sigma4"]:
            args += ";sigma4=%g" % c["sigma4"]
        return Plugin(args, fmt, c, host, frames)
    frames = c.get("frames", {"step": 32, "labels": 1}.get(kind))
    src = planes(c, frames, seed)
    fmt = nf.make_format(c["family"], c["bits"], c["float"], c["ssw"], c["ssh"])
    engines = [nf.Engine(params(c), fmt, c["width"], c["height"], frames, p) for p in range(len(src))]
    s = {"case": c, "src": src, "engines": engines, "stream": stream()}
    if kind == "labels":
        geo = engines[0].geometry()
        s["out"] = torch.empty((geo["nox"] * geo["noy"], c["bh"], geo["outwidth"]), device=DEV)
        return s
    s["dst"] = dst = [torch.zeros_like(p) for p in src]
    for e in engines:
        if c["dft"]:
            e.set_dft(1)
    if c["hidden"]:
        top = 1.0 if c["float"] else (1 << c["bits"]) - 1
        level = math.log((c["sigma"] * top / 255.0) ** 2 * c["bw"] * c["bh"])
        s["mlp"] = network(c["bh"] * (c["bw"] // 2 + 1), c["hidden"], 64, level, seed)
        for e in engines:
            nl.set_learned(e, s["mlp"])
    tables = [(e, 0, frames, [f.data_ptr() for f in p], p.stride(1) * p.element_size(), [f.data_ptr() for f in q],
               q.stride(1) * q.element_size()) for e, p, q in zip(engines, src, dst)]
    if kind == "step":
        s["arr"] = arr = (nf.RunItem * len(tables))()
        s["keep"] = keep = []
        for k, (e, _, _, sp, ss, dp, ds) in enumerate(tables):
            a, b = (ctypes.c_void_p * frames)(*sp), (ctypes.c_void_p * frames)(*dp)
            keep += [a, b]
            arr[k] = nf.RunItem(e.h, 0, 1, ctypes.cast(a, ctypes.POINTER(ctypes.c_void_p)), ss, ctypes.cast(b, ctypes.POINTER(ctypes.c_void_p)), ds)
        s["err"] = ctypes.create_string_buffer(512)
        s["next"], s["frames"] = 0, frames
    else:
        s["items"] = tables
    torch.cuda.synchronize()
    return s


class FramePlanes(ctypes.Structure):
    _fields_ = [("n", ctypes.c_int), ("data", ctypes.c_void_p * 4), ("stride", ctypes.c_int * 4)]


class Plugin:
    """The filter interface as a host application drives it: request_frames(n), then get_frame(n)."""

    def __init__(self, args, fmt, c, host, frames):
        L = nf.lib()
        L.nf3d_filter_get_frame.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p,
                                            ctypes.c_char_p, ctypes.c_size_t]
        self.case, self.host, self.frames, self.at = c, host, frames, 0
        self.h, self.err = ctypes.c_void_p(), ctypes.create_string_buffer(512)
        if L.nf3d_filter_create(args.encode(), ctypes.byref(fmt), c["width"], c["height"], frames, ctypes.byref(self.h), self.err, 512):
            raise RuntimeError(self.err.value.decode())
        self.refs = []
        for n in range(frames):
            f = FramePlanes(n=n)
            for p, a in enumerate(host):
                f.data[p], f.stride[p] = a[n].ctypes.data, a.strides[1]
            self.refs.append(f)
        self.outs = [np.zeros_like(a[0]) for a in host]
        self.dst = (ctypes.c_void_p * 4)(*[o.ctypes.data for o in self.outs])
        self.strides = (ctypes.c_int * 4)(*[o.strides[0] for o in self.outs])
        self.req = (ctypes.c_int * 8)()

    def get_frame(self, n):
        L = nf.lib()
        k = L.nf3d_filter_request_frames(self.h, n, self.req, 8)
        fr = (FramePlanes * k)(*[self.refs[self.req[i]] for i in range(k)])
        if L.nf3d_filter_get_frame(self.h, n, fr, k, self.dst, self.strides, self.err, 512):
            raise RuntimeError(self.err.value.decode())
        return self.outs

    def __del__(self):
        if self.h:
            nf.lib().nf3d_filter_destroy(self.h)


# ------------------------------------------------------------------ passes
def run(s):
    if isinstance(s, Plugin):
        n, s.at = s.at, (s.at + 1) % s.frames
        return s.get_frame(n)
    kind = s["case"]["kind"]
    if kind == "clip":
        nf.run_device_batch(s["items"], s["stream"])
        return s["dst"]
    if kind == "step":
        n = s["next"]
        s["next"] = (n + 1) % s["frames"]
        for it in s["arr"]:
            it.first = n
        if nf.lib().nf3d_run_device_batch(s["arr"], len(s["arr"]), ctypes.c_void_p(s["stream"]), s["err"], 512):
            raise RuntimeError(s["err"].value.decode())
        return [d[n] for d in s["dst"]]
    if kind == "labels":
        p = s["src"][0]
        s["engines"][0].region_psd(p.data_ptr(), p.stride(1) * 4, s["case"]["rx"], s["case"]["ry"], s["out"].data_ptr(), s["stream"])
        return s["out"]
    if kind == "dft2d":
        L, n, nb = nf.lib(), s["case"]["n"], s["case"]["blocks"]
        f = L.nf3d_dft2d_mfma
        f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_float, ctypes.c_void_p]
        if f(s["x"].data_ptr(), s["z"].data_ptr(), nb, n, 0, 1.0, s["stream"]) or f(s["z"].data_ptr(), s["y"].data_ptr(), nb, n, 1, 2.0 ** -8, s["stream"]):
            raise RuntimeError("nf3d_dft2d_mfma failed")
        return s["z"], s["y"]
    loss = s["mlp"].grad(s["x"].data_ptr(), s["t"].data_ptr(), s["case"]["batch"], s["stream"])
    return loss, s["mlp"].get_grads()


def work(case):
    if case["kind"] == "dft2d":
        n, nb = case["n"], case["blocks"]
        fft = 2.5 * n * n * math.log2(n * n)
        return {"bytes": nb * 2 * (4 * n * n + 8 * n * (n // 2 + 1)), "flops": nb * 2 * fft}
    if case["kind"] == "grad":
        d, h, n = case["d"], case["hidden"], case["batch"]
        p = 2 * d * h + h * h
        return {"bytes": 6 * n * d + 6 * p, "flops": 2.0 * n * (3 * p - d * h)}
    c = full(case)
    frames = c.get("frames", 1)
    bps = 4 if c["float"] else 1 if c["bits"] == 8 else 2
    by = fl = 0.0
    for w, h in plane_dims(c):
        nb = (-(-(w - c["ow"]) // (c["bw"] - c["ow"])) + 2) * (-(-(h - c["oh"]) // (c["bh"] - c["oh"])) + 2)
        el = c["bh"] * (c["bw"] // 2 + 1)
        fft = 2.5 * c["bw"] * c["bh"] * math.log2(c["bw"] * c["bh"])
        if c["kind"] == "labels":
            by += w * h * bps + nb * el * 4
            fl += nb * (fft + 8 * el)
            continue
        by += 2 * w * h * bps * frames
        fl += frames * nb * (2 * fft + el * 14 * max(1, c["bt"]))
        if c["bt"] == 0:  # the recursion's state, read and written once a call
            by += 2 * 3 * 8 * nb * el
        if c["hidden"]:  # one prediction in 16 frames
            fl += -(-frames // 16) * nb * 2.0 * (2 * el * c["hidden"] + c["hidden"] ** 2)
    return {"bytes": by, "flops": fl}


# ------------------------------------------------------------------ 64 bits
class Exact:
    """The filter on float planes in 64 bits: windows, overlapped blocks, gains, overlap-add."""

    def __init__(self, c, w, h):
        self.c, self.w, self.h = c, w, h
        f64 = dict(dtype=torch.float64, device=DEV)
        bw, bh, ow, oh = c["bw"], c["bh"], c["ow"], c["oh"]
        self.nox, self.noy = -(-(w - ow) // (bw - ow)) + 2, -(-(h - oh) // (bh - oh)) + 2

        def window(n, o):
            v = torch.ones(n, **f64)
            i = torch.arange(o, **f64)
            v[:o] = torch.cos(math.pi * (i - o + 0.5) / (2 * o))
            v[n - o:] = torch.cos(math.pi * (i + 0.5) / (2 * o))
            return v

        self.win = window(bh, oh)[:, None] * window(bw, ow)[None, :]
        self.grid = torch.fft.rfft2(self.win)
        ky = torch.arange(bh, **f64)
        dy = torch.where(ky >= bh // 2, bh - ky, ky) / (bh // 2)
        kx = torch.arange(bw // 2 + 1, **f64) / (bw // 2)
        d2 = dy[:, None] ** 2 + kx[None, :] ** 2
        self.wsharp = 1 - torch.exp(-d2 / (2 * 0.3 ** 2))
        wd = torch.exp(-0.7 * d2 * 4) - torch.exp(-d2 * 4)
        self.wdehalo = wd / wd.max()
        f32 = lambda v: float(np.float32(v))  # noqa: E731
        n = bw * bh
        self.smin, self.smax, self.ht = (f32(4.0) / 255) ** 2 * n, (f32(20.0) / 255) ** 2 * n, 50.0 ** 2 * n
        self.sig = torch.full((bh, bw // 2 + 1), (f32(c["sigma"]) / 255) ** 2 * n, **f64)
        if c["sigma4"]:  # sigma, sigma2, sigma3 alike, another at the lowest frequencies
            s1, s4 = f32(c["sigma"]) / 255, f32(c["sigma4"]) / 255
            fy = (bh - 2 * (torch.arange(bh, **f64) - bh // 2).abs()) / bh
            fx = torch.arange(bw // 2 + 1, **f64) / (bw // 2 + 1)
            f = torch.sqrt((fx[None, :] ** 2 + fy[:, None] ** 2) / 2)
            f3, f2 = math.sqrt(0.5) / 4, math.sqrt(0.5) / 2
            s = torch.where(f < f3, s4 + (s1 - s4) * f / f3, torch.full_like(f, s1))
            self.sig = s * s * n
        self.pattern = bool(c["sigma4"])

    def rows(self):
        """Plane row of each row that is filtered (fields stacked, the second one upside down)."""
        if not self.c["interlaced"]:
            return torch.arange(self.h, device=DEV)
        half = torch.arange(self.h // 2, device=DEV)
        return torch.cat([2 * half, self.h - 1 - 2 * half])

    def spectra(self, plane):
        c = self.c
        sx, sy = c["bw"] - c["ow"], c["bh"] - c["oh"]

        def mirror(n, total, start):
            v = (torch.arange(total, device=DEV) - start).abs()
            return torch.where(v >= n, 2 * n - 2 - v, v)

        p = plane.double()[self.rows()]
        cover = p[mirror(self.h, self.noy * sy + c["oh"], sy)][:, mirror(self.w, self.nox * sx + c["ow"], sx)]
        blocks = cover.unfold(0, c["bh"], sy).unfold(1, c["bw"], sx)
        return torch.fft.rfft2(blocks * self.win).reshape(-1, c["bh"], c["bw"] // 2 + 1)

    def synth(self, spec):
        c = self.c
        sx, sy = c["bw"] - c["ow"], c["bh"] - c["oh"]
        b = torch.fft.irfft2(spec, s=(c["bh"], c["bw"])) * self.win
        H, W = self.noy * sy + c["oh"], self.nox * sx + c["ow"]
        b = b.reshape(self.noy * self.nox, -1).T[None]
        out = torch.nn.functional.fold(b, (H, W), (c["bh"], c["bw"]), stride=(sy, sx))[0, 0]
        plane = torch.empty((self.h, self.w), dtype=torch.float64, device=DEV)
        plane[self.rows()] = out[sy:sy + self.h, sx:sx + self.w]
        return plane.clamp(0.0, 1.0)

    def sharpen(self, psd):
        f = 1 + self.c["sharpen"] * self.wsharp * torch.sqrt(psd * self.smax / ((psd + self.smin) * (psd + self.smax)))
        return f * (psd + self.ht) / ((psd + self.ht) + self.c["dehalo"] * self.wdehalo * psd)

    def mean_part(self, x):
        return self.c["degrid"] * x[:, :1, :1].real / self.grid[0, 0].real * self.grid

    def sharp_pass(self, x):
        if not self.c["sharpen"] and not self.c["dehalo"]:
            return x
        g = self.mean_part(x)
        d = x - g
        return d * self.sharpen(d.abs() ** 2 + 1e-15) + g

    def wiener(self, window, cur):
        """Frames of the window (oldest first), the current one's index."""
        n = len(window)
        g = self.mean_part(window[cur]) * n
        r = g.clone()
        for k in range(n):
            f = sum(v * complex(math.cos(2 * math.pi * k * (t - cur) / n), -math.sin(2 * math.pi * k * (t - cur) / n)) for t, v in enumerate(window))
            if k == 0:
                f = f - g
            psd = f.real ** 2 + f.imag ** 2 + 1e-15
            gain = ((psd - n * self.sig) / psd).clamp_min(0.0)
            if n == 1 and not self.pattern:
                gain = gain * self.sharpen(psd)
            r = r + f * gain
        r = r / n
        return r if n == 1 and not self.pattern else self.sharp_pass(r)

    def clip(self, frames):
        c, bt, n = self.c, self.c["bt"], len(frames)
        out, spec, state = [], {}, None
        for k in range(n):
            if bt == 0:
                if k == 0:
                    out.append(frames[0].double())
                    continue
                x = self.spectra(frames[k])
                if state is None:
                    one = self.sig if not self.pattern else torch.full_like(self.sig, (float(np.float32(c["sigma"])) / 255) ** 2 * c["bw"] * c["bh"])
                    z = torch.zeros_like(x)
                    state = (z, one * torch.ones_like(x.real) * (1 + 1j), one * torch.ones_like(x.real) * (1 + 1j))
                last, cov, proc = state
                sig = self.sig.clamp_min(1e-15)
                reset = ((x - last).real ** 2 > sig * 4) | ((x - last).imag ** 2 > sig * 4)
                s = cov + proc
                gain = torch.complex(s.real / (s.real + sig), s.imag / (s.imag + sig))
                full_sig = torch.complex(sig, sig)
                proc = torch.where(reset, full_sig, torch.complex(gain.real ** 2 * sig, gain.imag ** 2 * sig))
                cov = torch.where(reset, full_sig, torch.complex((1 - gain.real) * s.real, (1 - gain.imag) * s.imag))
                y = torch.where(reset, x, torch.complex(gain.real * x.real + (1 - gain.real) * last.real, gain.imag * x.imag + (1 - gain.imag) * last.imag))
                state = (y, cov, proc)
                out.append(self.synth(self.sharp_pass(y)))
                continue
            lo, hi = (k - bt // 2, k + (bt - 1) // 2) if bt > 1 else (k, k)
            if lo < 0 or hi >= n:
                lo = hi = k
            for i in list(spec):
                if i < lo - 1:
                    del spec[i]
            for i in range(lo, hi + 1):
                if i not in spec:
                    spec[i] = self.spectra(frames[i])
            window = [spec[i] for i in range(lo, hi + 1)]
            out.append(self.synth(self.wiener(window, k - lo) if bt > 0 else self.sharp_pass(window[0])))
        return torch.stack(out)

    def labels(self, plane, rx, ry):
        x = self.spectra(plane)
        d = x - self.mean_part(x)
        c = self.c
        fy = torch.arange(c["bh"], device=DEV, dtype=torch.float64)
        fy = torch.minimum(fy, c["bh"] - fy) * 2 / c["bh"]
        fx = torch.arange(c["bw"] // 2 + 1, device=DEV, dtype=torch.float64) * 2 / c["bw"]
        f2 = fy[:, None] ** 2 + fx[None, :] ** 2
        pat = (d.real ** 2 + d.imag ** 2) * (f2 / (f2 + 0.1 ** 2))
        sums = pat.sum((1, 2)).reshape(self.noy, self.nox).cpu()
        sums[:2], sums[-2:], sums[:, :2], sums[:, -2:] = 3e38, 3e38, 3e38, 3e38

        def first_min(y0, y1, x0, x1):
            v = sums[y0:y1, x0:x1]
            i = int(torch.argmin(v.reshape(-1)))
            return (y0 + i // v.shape[1]) * self.nox + x0 + i % v.shape[1] if float(v.reshape(-1)[i]) < 1e15 else None

        whole = first_min(0, self.noy, 0, self.nox)
        pick = torch.empty((self.noy, self.nox), dtype=torch.int64)
        for y0 in range(0, self.noy, ry):
            for x0 in range(0, self.nox, rx):
                best = first_min(y0, min(y0 + ry, self.noy), x0, min(x0 + rx, self.nox))
                pick[y0:y0 + ry, x0:x0 + rx] = whole if best is None else best
        return pat[pick.reshape(-1).to(DEV)]


def exact(case, seed):
    kind = case["kind"]
    if kind == "dft2d":
        s = prepare(case, seed)
        x = s["x"].double()
        return torch.view_as_real(torch.fft.rfft2(x)), x * case["n"] ** 2
    if kind == "grad":
        s = prepare(case, seed)
        d, h = case["d"], case["hidden"]
        flat = torch.from_numpy(nl.init_params(d, h, d, seed, out_bias=_bias(d, 9.0, seed))).to(DEV)
        sizes = [(d, h), (h,), (h, h), (h,), (h, d), (d,)]
        w, at = [], 0
        for sz in sizes:  # the matrices as the 16-bit values that the products take
            n = math.prod(sz)
            v = flat[at:at + n].reshape(sz)
            w.append((v.to(torch.bfloat16) if len(sz) == 2 else v).double().requires_grad_())
            at += n
        a = s["x"].double()
        a = torch.nn.functional.gelu(a @ w[0] + w[1])
        a = torch.nn.functional.gelu(a @ w[2] + w[3])
        y = a @ w[4] + w[5]
        loss = (y + s["t"].double() * torch.exp(-y)).mean()
        loss.backward()
        return loss.detach().reshape(()), torch.cat([v.grad.reshape(-1) for v in w])
    c = full(case)
    if not c["float"] or kind in ("plugin", "step") or c["hidden"]:
        return None  # samples of integer formats; a float frame at a time is the same as a clip of it; the network's own case is "grad"
    if kind == "labels":
        return Exact(c, c["width"], c["height"]).labels(planes(c, 1, seed)[0][0], c["rx"], c["ry"])
    return [Exact(c, p.shape[2], p.shape[1]).clip(p) for p in planes(c, c["frames"], seed)]


def _bias(d, level, seed):
    """The output bias that ``network`` draws after its input normalisation."""
    rng = np.random.default_rng(seed)
    rng.standard_normal(d)
    return level + 0.2 * rng.standard_normal(d)
