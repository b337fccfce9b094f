"""What a program has this library do, as cases that can be timed.

Four ways in, each the whole call as a program makes it -- a context is good
for one image (iw_process_image refuses a second use), so every pass sets up
its own:

  device  iwamd_process_device_noalloc: input and output in the program's
          device memory (a GPU pipeline's resize step)
  host    api.Library.run, i.e. iw_process_image: host bytes in, the finished
          image's host bytes out (the drop-in use of the C API)
  batch   api.Library.run_batch: many images of uneven sizes in one device
          block and one graph launch (making thumbnails, dataset preparation)
  serve   api.Server: requests queued on a running request loop, results taken
          when all are done (image serving)

Pixels are the synthetic recipes of imageworsener_amd/synth.py, drawn with
torch: `scene` is the left gradient, right noise with hard blocks; `texture`
three sinusoid gratings plus noise; `radial` a noisy radial ramp; alpha comes
in constant tiles, a tenth of them fully transparent.
"""
import ctypes
import math

import numpy as np
import torch

from imageworsener_amd import api

RADIUS = {"triangle": 1.0, "catrom": 2.0, "mitchell": 2.0, "lanczos2": 2.0, "lanczos3": 3.0}
PROFILE_FLOAT = api.PROFILE_PNG | 0x4000  # IW_PROFILE_HDRI: 32-bit float output
SAMPLETYPE_FLOAT = 1
BATCH_FILTERS = ["triangle", "catrom", "lanczos2", "lanczos3"]
SERVE_FILTERS = ["lanczos3", "mitchell"]
MiB = 1 << 20


# ---- the cases -----------------------------------------------------------------

def _image(call, ch, depth, w, h, ow, oh, filt, dither="none", colors=0, out_depth=8, form="plain", name=None):
    c = {"call": call, "ch": ch, "depth": depth, "w": w, "h": h, "ow": ow, "oh": oh, "filter": filt,
         "dither": dither, "colors": colors, "out_depth": out_depth, "form": form}
    if name:
        c["name"] = name
    return c


def _many(call, images, lo, hi, list_seed, form="plain", name=None):
    c = {"call": call, "images": images, "lo": lo, "hi": hi, "list_seed": list_seed, "form": form}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # An icon halved: nothing but the cost of a call.
        _image("device", "RGBA", 8, 64, 48, 32, 24, "lanczos3", name="device-icon"),
        # The plain 640x480 to 320x240 preview, on host bytes.
        _image("host", "RGB", 8, 640, 480, 320, 240, "lanczos3", name="host-preview"),
        # A 12-megapixel camera picture to a page-sized one, on the device.
        _image("device", "RGB", 8, 4000, 3000, 1000, 750, "lanczos3", name="device-photo"),
        # 16-bit RGBA artwork reduced to 8 bits with Floyd-Steinberg, on the device.
        _image("device", "RGBA", 16, 2047, 2048, 1000, 1001, "mitchell", dither="f", name="device-rgba16-fs"),
        # An RGBA picture enlarged with the chosen-precision (MFMA) form.
        _image("device", "RGBA", 8, 1024, 768, 2048, 1536, "catrom", form="fast", name="device-enlarge-fast"),
        # Linear float pixels (HDR) in and out.
        _image("device", "RGB", 32, 1023, 767, 512, 384, "catrom", out_depth=32, name="device-float"),
        # The 4096x4096 16-bit RGBA image to 1000x1000, Floyd-Steinberg, host bytes.
        _image("host", "RGBA", 16, 4096, 4096, 1000, 1000, "mitchell", dither="f", name="host-rgba16-fs"),
        # 2048x2048 16-bit linear grey enlarged to 3072x3072 in 4 grey levels: error diffusion, then random dither.
        _image("host", "GRAY", 16, 2048, 2048, 3072, 3072, "catrom", dither="jjn", colors=4, name="host-grey-jjn"),
        _image("host", "GRAY", 16, 2048, 2048, 3072, 3072, "catrom", dither="r", colors=4, name="host-grey-random"),
        # Uneven RGBA images, sides 64 to 1024, each with its own scales and filter; both forms.
        _many("batch", 48, 64, 1024, 4, name="batch-plain"),
        _many("batch", 64, 64, 1024, 5, form="fast", name="batch-fast"),
        # Requests of 8- and 16-bit RGB pictures, 8-bit Floyd-Steinberg results.
        _many("serve", 12, 256, 2048, 5, name="serve"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _scratch(c):
    """About the device memory a device call takes besides its buffers: its
    64 MiB array holds the FP32 intermediate and the diffusion samples."""
    nch = api.NCH[api.IMGTYPE[c["ch"]]]
    inter = 4 * nch * c["oh"] * c["w"] if c["w"] > 2048 or c["form"] == "fast" else 0
    ed = 8 * nch * c["ow"] * (c["oh"] + 12) if c["dither"] not in ("none", "o", "r") else 0
    return inter + ed


def draw(rng):
    call = rng.choices(["device", "host", "batch", "serve"], [5, 3, 1, 1])[0]
    if call == "batch":
        return _many("batch", rng.randint(16, 64), 64, 1024, rng.randrange(1 << 20), rng.choice(["plain", "fast"]))
    if call == "serve":
        return _many("serve", rng.randint(4, 12), 256, 2048, rng.randrange(1 << 20))
    while True:
        w, h = _log(rng, 48, 4096), _log(rng, 48, 4096)
        sx = rng.uniform(0.2, 1.0) if rng.random() < 0.7 else rng.uniform(1.0, 2.0)
        sy = sx if rng.random() < 0.7 else sx * rng.uniform(0.8, 1.25)
        c = _image(call, rng.choices(["RGB", "RGBA", "GRAY"], [5, 4, 2])[0], rng.choices([8, 16], [2, 1])[0], w, h,
                   max(1, round(w * sx)), max(1, round(h * sy)), rng.choice(sorted(RADIUS)))
        kind = rng.random()
        if kind < 0.12:
            c.update(depth=32, out_depth=32, ch="RGB")
        elif kind < 0.30:
            c["out_depth"] = 16
        elif kind < 0.65:
            c["dither"] = rng.choice(["f", "f", "f", "jjn", "sierra", "atkinson", "o", "r"])
            if rng.random() < 0.3:
                c["colors"] = rng.choice([2, 4, 6, 16])
        if c["depth"] != 32 and c["dither"] in ("none", "o") and rng.random() < 0.35:
            c["form"] = "fast"
        # Device calls fit their scratch array; nothing is larger than the listed ones.
        if c["ow"] * c["oh"] > 2500 * 2500 or max(c["ow"], c["oh"]) > 3072:
            continue
        if call == "device" and _scratch(c) > 56 * MiB:
            continue
        return c


# ---- inputs ----------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda" if torch.cuda.is_available() else "cpu")
    g.manual_seed(seed & 0x7FFFFFFF)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=g.device, dtype=torch.float32)


def _texture(g, h, w, n):
    size = float(max(w, h))
    xs = torch.arange(w, device=g.device, dtype=torch.float32)
    ys = torch.arange(h, device=g.device, dtype=torch.float32)
    out = torch.empty(h, w, n, device=g.device)
    for k in range(n):
        v = torch.full((h, w), 0.5, device=g.device)
        for f, th, ph in _rand(g, 3, 3).tolist():
            a = 2 * math.pi * (1 + 255 * f) / size
            ax, by = a * math.cos(th * math.pi) * xs + 2 * math.pi * ph, a * math.sin(th * math.pi) * ys
            v += (torch.sin(by)[:, None] * torch.cos(ax) + torch.cos(by)[:, None] * torch.sin(ax)) / 6
        out[..., k] = v + (_rand(g, h, w) - 0.5) / 16
    return out.clamp_(0, 1)


def _scene(g, h, w, n):
    corner = _rand(g, 4, n)
    fx = torch.linspace(0, 1, w, device=g.device)[None, :, None]
    fy = torch.linspace(0, 1, h, device=g.device)[:, None, None]
    out = (corner[0] * ((1 - fx) * (1 - fy)) + corner[1] * (fx * (1 - fy)) + corner[2] * ((1 - fx) * fy) +
           corner[3] * (fx * fy))
    half = w // 2
    out[:, half:] = _rand(g, h, w - half, n)
    bh, bw = (h + 15) // 16, (w - half + 15) // 16
    coin = _rand(g, bh, bw) < 0.5
    odd = (torch.arange(bh, device=g.device)[:, None] + torch.arange(bw, device=g.device)) % 2
    block = torch.where(coin, 1.0 - odd, torch.full_like(odd, -1.0, dtype=torch.float32))
    block = block.repeat_interleave(16, 0).repeat_interleave(16, 1)[:h, :w - half, None]
    out[:, half:] = torch.where(block >= 0, block, out[:, half:])
    return out


def _radial(g, h, w):
    y = torch.arange(h, device=g.device) - (h - 1) / 2
    x = torch.arange(w, device=g.device) - (w - 1) / 2
    r = torch.sqrt(y[:, None] ** 2 + x ** 2) / math.sqrt((h * h + w * w) / 4)
    return (r + (_rand(g, h, w) - 0.5) / 64).clamp_(0, 1)[..., None]


def _pixels(ch, depth, w, h, seed, kind):
    """Samples (h, w, channels): uint8 for 8 and 16 bits (big-endian pairs), float32 for 32."""
    g = _gen(seed)
    if ch == "GRAY":
        v = _radial(g, h, w)
    else:
        v = (_texture if kind == "texture" else _scene)(g, h, w, 3)
    if ch == "RGBA":
        t = 64 if w * h > 1 << 20 else 16
        a = _rand(g, (h + t - 1) // t, (w + t - 1) // t)
        a = torch.where(_rand(g, *a.shape) < 0.1, torch.zeros_like(a), a)
        a = a.repeat_interleave(t, 0).repeat_interleave(t, 1)[:h, :w, None]
        v = torch.cat([v, a], 2)
    if depth == 32:
        return v.contiguous()
    if depth == 8:
        return (v * 255 + 0.5).to(torch.uint8)
    q = (v * 65535 + 0.5).to(torch.int32).clamp_(0, 65535)
    return torch.stack([q >> 8, q & 255], -1).to(torch.uint8).reshape(h, w, -1).contiguous()


def _kind(c):
    return "texture" if c["depth"] == 16 or c["w"] * c["h"] > 1 << 21 else "scene"


def _settings(c):
    """The job's settings (api.image_job's keywords)."""
    s = {"canvas": (c["ow"], c["oh"]), "resize": api.resize_both(c["filter"]),
         "profile": PROFILE_FLOAT if c["out_depth"] == 32 else api.PROFILE_PNG}
    if c["out_depth"] == 16 or (c["out_depth"] == 8 and c["depth"] == 16):
        s["depth"] = c["out_depth"]
    if c["ch"] == "GRAY" and c["depth"] == 16 or c["depth"] == 32:
        s["input_cs"] = (api.CS["linear"], 0.0)
    if c["depth"] == 32:
        s["output_cs"] = (api.CS["linear"], 0.0)
    if c["dither"] != "none":
        s["dither"] = [(api.CH_ALL,) + api.DITHER[c["dither"]]]
        if c["dither"] == "r":
            s["random_seed"] = 3
    if c["colors"]:
        s["color_count"] = [(api.CH_ALL, c["colors"])]
    if c["form"] == "fast":
        s["precision"] = api.PRECISION_FAST
    return s


def _job(c, pixels):
    job = api.image_job(pixels.cpu().numpy().view(np.uint8), c["w"], c["h"], api.IMGTYPE[c["ch"]], c["depth"],
                        **_settings(c))
    if c["depth"] == 32:
        job["image"]["sampletype"] = SAMPLETYPE_FLOAT
    return job


def _list(c):
    """The images of a batch or a run of requests, as single cases."""
    r = np.random.default_rng(c["list_seed"])
    lo, hi = math.log(c["lo"]), math.log(c["hi"])
    out = []
    for _ in range(c["images"]):
        w, h = (int(round(math.exp(v))) for v in r.uniform(lo, hi, 2))
        if c["call"] == "batch":
            sx, sy = r.uniform(0.25, 2.0, 2)
            filt, ch, depth, dither = BATCH_FILTERS[r.integers(4)], "RGBA", 8, "none"
        else:
            sx = sy = r.uniform(0.1, 1.5)
            filt, ch, depth, dither = SERVE_FILTERS[r.integers(2)], "RGB", int(r.choice([8, 16])), "f"
        out.append(_image("host", ch, depth, w, h, max(1, round(w * sx)), max(1, round(h * sy)), filt, dither,
                          form=c["form"]))
    return out


# ---- what a program holds ----------------------------------------------------------

_held = {}


def _library():
    if "lib" not in _held:
        lib = api.Library()
        fn = lib.dll.iwamd_process_device_noalloc
        fn.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_void_p, ctypes.c_size_t,
                       ctypes.c_void_p, ctypes.POINTER(api.Image)]
        fn.restype = ctypes.c_int
        _held["lib"] = lib
    return _held["lib"]


def _server():
    """One request loop for the life of the program."""
    if "server" not in _held:
        _held["server"] = api.Server(_library(), streams=4)
    return _held["server"]


def prepare(case, seed):
    state = {"case": case, "lib": _library()}
    if case["call"] in ("batch", "serve"):
        state["jobs"] = [_job(c, _pixels(c["ch"], c["depth"], c["w"], c["h"], seed * 131 + k,
                                         "scene" if case["call"] == "batch" else "texture"))
                         for k, c in enumerate(_list(case))]
        if case["call"] == "serve":
            state["server"] = _server()
        return state
    px = _pixels(case["ch"], case["depth"], case["w"], case["h"], seed, _kind(case))
    if case["call"] == "host":
        state["job"] = _job(case, px)
        return state
    nch = api.NCH[api.IMGTYPE[case["ch"]]]
    img = api.Image()
    img.imgtype = api.IMGTYPE[case["ch"]]
    img.bit_depth = case["depth"]
    img.sampletype = SAMPLETYPE_FLOAT if case["depth"] == 32 else 0
    img.width, img.height = case["w"], case["h"]
    img.bpr = case["w"] * nch * case["depth"] // 8
    state.update(image=img, settings=_settings(case), d_in=px.reshape(-1),
                 d_out=torch.empty(case["ow"] * case["oh"] * nch * (case["out_depth"] // 8), dtype=torch.uint8,
                                   device=px.device))
    return state


def _run_device(s):
    lib = s["lib"]
    d = lib.dll
    ctx = d.iw_create_context(None)
    try:
        d.iw_set_input_image(ctx, ctypes.byref(s["image"]))
        lib._setup(ctx, s["settings"])
        stream = torch.cuda.current_stream().cuda_stream
        d_in, d_out = s["d_in"], s["d_out"]
        if not d.iwamd_process_device_noalloc(ctx, d_in.data_ptr(), d_in.numel() * d_in.element_size(),
                                              d_out.data_ptr(), d_out.numel(), stream, None):
            buf = ctypes.create_string_buffer(300)
            raise RuntimeError(d.iw_get_errormsg(ctx, buf, 300).decode(errors="replace"))
    finally:
        d.iw_destroy_context(ctx)
    return d_out.view(torch.float32) if s["case"]["out_depth"] == 32 else d_out


def _bytes(results, case):
    for r in results:
        if not r["ok"]:
            raise RuntimeError(r["error"])
    out = [r["pixels"] for r in results]
    return [p.view(np.float32) for p in out] if case.get("out_depth") == 32 else out


def run(state):
    case, lib = state["case"], state["lib"]
    if case["call"] == "device":
        return _run_device(state)
    if case["call"] == "host":
        return _bytes([lib.run(state["job"])], case)[0]
    if case["call"] == "batch":
        return _bytes(lib.run_batch(state["jobs"]), case)
    srv = state["server"]
    for job in state["jobs"]:
        srv.submit(job)
    out = srv.results()
    # The finished requests' contexts go; the loop stays for the next ones.
    for ctx in srv.ctxs:
        lib.dll.iw_destroy_context(ctx)
    srv.ctxs, srv.ids = [], []
    return _bytes(out, case)


# ---- the work, and the exact values -------------------------------------------------

def work(case):
    """Input and output image once; a multiply and an add per tap of both
    resampling passes (vertical first, over the input's columns)."""
    if case["call"] in ("batch", "serve"):
        each = [work(c) for c in _list(case)]
        return {k: sum(e[k] for e in each) for k in ("bytes", "flops")}
    nch = api.NCH[api.IMGTYPE[case["ch"]]]
    w, h, ow, oh = (case[k] for k in ("w", "h", "ow", "oh"))
    tv, th = (2 * RADIUS[case["filter"]] * max(1.0, a / b) for a, b in ((h, oh), (w, ow)))
    return {"bytes": nch * (w * h * case["depth"] + ow * oh * case["out_depth"]) / 8,
            "flops": 2.0 * nch * (tv * w * oh + th * ow * oh)}


def _filter(name, x):
    x = np.abs(x)
    if name == "triangle":
        return np.maximum(0.0, 1.0 - x)
    if name in ("lanczos2", "lanczos3"):
        return np.where(x < RADIUS[name], np.sinc(x) * np.sinc(x / RADIUS[name]), 0.0)
    b, c = (0.0, 0.5) if name == "catrom" else (1 / 3, 1 / 3)
    near = ((12 - 9 * b - 6 * c) * x ** 3 + (-18 + 12 * b + 6 * c) * x ** 2 + (6 - 2 * b)) / 6
    far = ((-b - 6 * c) * x ** 3 + (6 * b + 30 * c) * x ** 2 + (-12 * b - 48 * c) * x + (8 * b + 24 * c)) / 6
    return np.where(x < 1, near, np.where(x < 2, far, 0.0))


def _matrix(name, n_in, n_out):
    pos = (np.arange(n_out) + 0.5) * n_in / n_out - 0.5
    m = _filter(name, (np.arange(n_in) - pos[:, None]) / max(1.0, n_in / n_out))
    return m / m.sum(1, keepdims=True)


def exact(case, seed):
    """Linear float images have a value in 64 bits; the others are whole numbers."""
    if case.get("out_depth") != 32:
        return None
    px = _pixels(case["ch"], 32, case["w"], case["h"], seed, _kind(case)).cpu().numpy().astype(np.float64)
    mv, mh = _matrix(case["filter"], case["h"], case["oh"]), _matrix(case["filter"], case["w"], case["ow"])
    out = np.stack([mv @ px[..., k] @ mh.T for k in range(px.shape[2])], 2)
    return out.reshape(-1)
