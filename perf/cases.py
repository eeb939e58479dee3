"""Performance cases of the ray march: what a program that renders with this
package has it do, over the ranges it is used in.

listed() gives the named cases, draw(rng) one more of the same ranges,
prepare(case, seed) what a program holds before the call, run(state) one pass
through the public entry points, work(case) the bytes and operations a pass
cannot do without, exact(case, seed) the same result in 64 bits from plain
torch.

Kinds of case:
  frame    camera -> entry/exit points -> one frame, all buffers on the device
  edit     a transfer-function edit in pre-integrated mode: new TF, new
           pre-integration table on the device, one frame
  host     one frame through host buffers with its statistics, as the
           HIPRaycaster processor renders it
  jobs     many uneven volumes, each with its own TF and camera, one launch
  views    several views of one volume in one launch
  learned  one frame with learned stepping (judge and fallback included)
  train    Adam steps of the stepping network on one minibatch
"""
import math
import random

import numpy as np
import torch

from voreen_amd import hipdvr as H
from voreen_amd import workloads as W

MODES = {"dvr": H.COMPOSITE_DVR, "mip": H.COMPOSITE_MIP, "mop": H.COMPOSITE_MOP, "mida": H.COMPOSITE_MIDA,
         "iso": H.COMPOSITE_ISO, "fhp": H.COMPOSITE_FHP, "fhn": H.COMPOSITE_FHN}
LIGHT = dict(pos=(2.3, 1.5, 1.5), ambient=0.4, diffuse=0.8, specular=0.6, shininess=60.0)
LEARNING_RATE = 2e-3


def _frame(kind, dims, dtype, image, content, mode="dvr", shading="none", classif="tf", filt="linear", table=0,
           rate=2.0, radius=3.5):
    return dict(kind=kind, x=dims[0], y=dims[1], z=dims[2], dtype=dtype, w=image[0], h=image[1], content=content,
                mode=mode, shading=shading, classif=classif, filter=filt, table=table, rate=rate, radius=radius)


def listed():
    return [
        # the smallest call: a thumbnail-sized preview of a small byte volume
        # (eight noisy blobs, random 4-key TF); latency and launches count
        dict(_frame("frame", (128, 128, 128), "u8", (256, 256), "blobs"), name="frame_128_u8"),
        # the interactive view of a 512^3 16-bit volume with Phong lighting
        dict(_frame("frame", (512, 512, 512), "u16", (1024, 1024), "shells", shading="phong"), name="frame_512_phong"),
        # maximum intensity projection of a CT-shaped 16-bit volume
        dict(_frame("frame", (512, 512, 361), "u16", (1024, 1024), "shells", mode="mip"), name="frame_mip"),
        # shaded iso surface of a ragged byte volume in an odd window
        dict(_frame("frame", (301, 257, 199), "u8", (811, 613), "turbulence", mode="iso", shading="phong"),
             name="frame_iso_ragged"),
        # pre-integrated classification of a ragged 16-bit volume, odd window
        dict(_frame("frame", (381, 255, 317), "u16", (1019, 763), "shells", classif="preint", table=256),
             name="frame_preint"),
        # dragging a TF key in pre-integrated mode: a new 1024^2 table per frame
        dict(_frame("edit", (256, 256, 256), "u8", (512, 512), "shells", classif="preint", table=1024),
             name="edit_preint_1024"),
        # the processor's frame: host entry/exit images in, host image out,
        # statistics read back
        dict(_frame("host", (256, 256, 256), "u16", (512, 512), "shells", shading="phong"), name="host_256_phong"),
        # 64 uneven volumes (64..384 voxels an axis, bytes or 16 bits) in one launch
        dict(kind="jobs", n=64, lo=64, hi=384, image=512, name="jobs_64"),
        # 12 orbit views of the 512^3 volume in one launch, Phong
        dict(_frame("views", (512, 512, 512), "u16", (1024, 1024), "shells", shading="phong"), n=12, name="views_12"),
        # the largest call: a 4K frame of a 1024^3 volume whose records pass 4 GiB
        dict(_frame("frame", (1024, 1024, 1024), "u16", (3840, 2160), "turbulence", shading="phong"),
             name="frame_1024_4k"),
        # learned stepping on the 512^3 volume
        dict(_frame("learned", (512, 512, 512), "u16", (1024, 1024), "shells", shading="phong"), name="learned_512"),
        # training the stepping network: 16 Adam steps on 8192 rows
        dict(kind="train", rows=8192, steps=16, name="train_8192"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 8 + ["edit", "host", "host", "jobs", "views", "learned", "train"])
    if kind == "train":
        return dict(kind="train", rows=_log(rng, 300, 16384), steps=rng.randint(4, 24))
    if kind == "jobs":
        return dict(kind="jobs", n=_log(rng, 6, 64), lo=48, hi=rng.randint(160, 384), image=_log(rng, 150, 512))
    dims = tuple(_log(rng, 64, 640) for _ in range(3))
    image = (_log(rng, 128, 1920), _log(rng, 128, 1200))
    dtype = rng.choice(["u8", "u16"])
    shading = rng.choice(["none", "phong"])
    rate = rng.choice([1.0, 2.0, 2.0, 3.0])
    radius = rng.uniform(2.2, 3.6)
    if kind == "frame":
        mode = rng.choice(["dvr"] * 5 + ["mip", "mip", "mop", "mida", "iso", "fhp", "fhn"])
        classif = rng.choice(["tf", "tf", "tf", "preint"]) if mode == "dvr" else "tf"
        filt = rng.choice(["linear"] * 7 + ["nearest"])
        if mode != "dvr" or classif != "tf":
            image, rate = (min(image[0], 1100), min(image[1], 900)), min(rate, 2.0)
        if mode in ("mip", "mida"):
            shading = "none"   # projections keep a maximum: their colour is the TF's
        content = rng.choice(["shells", "shells", "turbulence"])
        if mode in ("iso", "mop"):
            content = "turbulence"   # a smooth field: thin bands of alpha are surfaces there
        return _frame("frame", dims, dtype, image, content, mode, shading, classif, filt,
                      rng.choice([128, 255, 256, 511]) if classif == "preint" else 0, rate, radius)
    if kind == "edit":
        dims = tuple(min(d, 384) for d in dims)
        image = (min(image[0], 800), min(image[1], 800))
        return _frame("edit", dims, dtype, image, "shells", classif="preint", table=_log(rng, 128, 1024), rate=rate,
                      radius=radius)
    if kind == "host":
        return _frame("host", dims, dtype, (min(image[0], 1100), image[1]), "shells", shading=shading, rate=rate,
                      radius=radius)
    if kind == "views":
        return dict(_frame("views", dims, dtype, (min(image[0], 1024), min(image[1], 1024)), "shells",
                           shading=shading, rate=rate, radius=radius), n=rng.randint(2, 12))
    return _frame("learned", tuple(max(d, 160) for d in dims), dtype, (max(image[0], 400), max(image[1], 400)),
                  "shells", shading=shading, radius=radius)


# ---------------------------------------------------------------------------
# inputs, made on the GPU from the seed alone
# ---------------------------------------------------------------------------
def _rng(seed, what):
    return random.Random("%d/%s" % (seed, what))


def _grid(n, device):
    return (torch.arange(n, device=device, dtype=torch.float32) + 0.5) / n - 0.5


def _noise(gen, dims, octaves, base, device):
    """Sum of trilinearly interpolated random grids, amplitude halving, in [0, 1]."""
    x, y, z = dims
    f, amp, norm = torch.zeros((z, y, x), device=device), 1.0, 0.0
    for o in range(octaves):
        g = base << o
        cells = torch.rand((1, 1, min(g, z), min(g, y), min(g, x)), generator=gen, device=device)
        f += amp * torch.nn.functional.interpolate(cells, size=(z, y, x), mode="trilinear", align_corners=True)[0, 0]
        norm += amp
        amp *= 0.5
    return f / norm


def _volume(dims, dtype, content, seed):
    """Voxels as a (z, y, x) tensor of raw values in int32 (0..255 or 0..65535)."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed * 1000003 + 17)
    x, y, z = dims
    top = 255.0 if dtype == "u8" else 65535.0
    gx, gy, gz = _grid(x, dev), _grid(y, dev), _grid(z, dev)
    if content == "blobs":
        # eight Gaussian blobs plus uniform noise of +-2/255
        r = _rng(seed, "blobs")
        f = torch.zeros((z, y, x), device=dev)
        for _ in range(8):
            c, s, a = [r.uniform(-0.3, 0.3) for _ in range(3)], r.uniform(0.05, 0.15), r.uniform(0.3, 1.0)
            e = [torch.exp(-(g - m) ** 2 / (2 * s * s)) for g, m in zip((gx, gy, gz), c)]
            f += a * e[2][:, None, None] * e[1][None, :, None] * e[0][None, None, :]
        f = f / f.max() + torch.randint(-2, 3, f.shape, generator=gen, device=dev) / 255.0
    elif content == "shells":
        # nested ellipsoid shells of five densities with fBm noise in air
        rr = torch.sqrt((gx / 0.62)[None, None, :] ** 2 + (gy / 0.56)[None, :, None] ** 2 +
                        (gz / 0.50)[:, None, None] ** 2)
        f = torch.zeros_like(rr)
        for edge, d in ((1.0, 0.15), (0.85, 0.45), (0.70, 0.70), (0.50, 0.25), (0.30, 0.90)):
            f[rr < edge] = d
        f = torch.where(rr < 1.0, f + 0.05 * (2 * _noise(gen, dims, 4, 8, dev) - 1), torch.zeros_like(f))
    else:
        # fBm turbulence with its lower part cut to empty space
        f = _noise(gen, dims, 6, 6, dev)
        cut = torch.quantile(f.reshape(-1)[:: max(1, f.numel() // 1000000)][:1000000], 0.4)
        f = ((f - cut) / (f.max() - cut)).clamp_(min=0.0)
    return (f.clamp_(0.0, 1.0) * top + 0.5).floor_().clamp_(max=top).to(torch.int32)


def _keys(content, seed):
    """1D TF keys as (intensity, rgba) for the content."""
    r = _rng(seed, "keys")

    def col(a):
        return (r.randrange(256), r.randrange(256), r.randrange(256), a)

    if content == "blobs":
        return [(float(np.float32(i)), col(r.randrange(256)))
                for i in sorted(r.random() for _ in range(r.randint(4, 8)))]
    if content == "shells":
        a1, a2 = 40 + r.randrange(120), 80 + r.randrange(150)
        ks = [(0.0, 0), (0.42, 0), (0.50, a1), (0.58, 0), (0.86, 0), (1.0, a2)]
    else:
        ks = [(0.0, 0), (0.04, 0), (0.10, 12 + r.randrange(20)), (0.22, 4), (0.30, 60 + r.randrange(60)),
              (0.50, 140 + r.randrange(60)), (1.0, 255)]
    return [(float(np.float32(i)), col(a)) for i, a in ks]


def _lookup(keys, values):
    """Bytes of the keys' piecewise linear map at float32 values, channels truncated."""
    v = np.clip(np.asarray(values, np.float32), np.float32(0), np.float32(1))
    its = np.array([k[0] for k in keys], np.float32)
    cols = np.array([k[1] for k in keys], np.float32)
    hi = np.searchsorted(its, v, side="left")
    lo = np.clip(hi - 1, 0, len(keys) - 1)
    up = np.clip(hi, 0, len(keys) - 1)
    span = its[up] - its[lo]
    f = ((v - its[lo]) / np.where(span > 0, span, np.float32(1)))[:, None]
    out = cols[lo] + (cols[up] - cols[lo]) * f
    out = np.where((hi == 0)[:, None], cols[0], np.where((hi == len(keys))[:, None], cols[-1], out))
    return out.astype(np.uint8)


def _tf(keys, dtype):
    n = 256 if dtype == "u8" else 4096
    return _lookup(keys, np.arange(n, dtype=np.float32) / np.float32(n - 1))


def _camera(seed, radius, view=0, views=36):
    """Orbit camera of this seed (float32 values): eye, focus, up, fovy, near."""
    r = _rng(seed, "camera")
    th = 2.0 * math.pi * (r.random() + view / views)
    el = math.radians(r.uniform(-35.0, 45.0))
    eye = (radius * math.sin(th) * math.cos(el), radius * math.sin(el), radius * math.cos(th) * math.cos(el))
    return dict(eye=tuple(float(np.float32(v)) for v in eye), fovy=30.0, near=0.1)


def _box(dims):
    ext = np.array(dims, np.float64) / max(dims)
    return (-ext / 2).astype(np.float32), (ext / 2).astype(np.float32)


def _placed(dims):
    llf, urb = _box(dims)
    sp = tuple(float((urb[i] - llf[i]) / dims[i]) for i in range(3))
    return sp, tuple(float(llf[i] + 0.5 * sp[i]) for i in range(3))


def _dims(case):
    return (case["x"], case["y"], case["z"])


# ---------------------------------------------------------------------------
# states
# ---------------------------------------------------------------------------
class _State(dict):
    """What a program holds; its device objects are given back with it."""

    def __del__(self):
        for o in self.get("close", ()):
            o.close()


_context = None


def _ctx():
    global _context
    if _context is None:
        _context = H.Context(0)
    return _context


def _buffer(t):
    """A torch tensor's memory as the package's device buffer (the tensor owns it)."""
    b = H.DeviceBuffer(_ctx(), H.C.c_void_p(t.data_ptr()), t.numel() * t.element_size())
    b.tensor = t
    return b


def _image(w, h):
    return _buffer(torch.zeros((h, w, 4), dtype=torch.float32, device="cuda"))


def _device_volume(dims, dtype, content, seed, **kw):
    raw = _volume(dims, dtype, content, seed)
    if dtype == "u8":
        vox = raw.to(torch.uint8)
    else:
        vox = torch.where(raw > 32767, raw - 65536, raw).to(torch.int16)   # the same 16 bits
    del raw
    torch.cuda.synchronize()
    v = _ctx().volume_device(_buffer(vox), dims, H.U8 if dtype == "u8" else H.U16, **kw)
    _ctx().synchronize()
    return v


def _device_camera(cam):
    c = H.Camera()
    c.eye[:] = list(cam["eye"])
    c.focus[:] = [0.0, 0.0, 0.0]
    c.up[:] = [0.0, 1.0, 0.0]
    c.fovy_deg, c.near_dist = cam["fovy"], cam["near"]
    return c


def _params(case, cam):
    return H.default_params(W.step_for(_dims(case), case["rate"]),
                            filter_=H.FILTER_NEAREST if case["filter"] == "nearest" else H.FILTER_LINEAR,
                            classification=H.CLASS_PREINT if case["classif"] == "preint" else H.CLASS_TF,
                            shading=H.SHADE_PHONG if case["shading"] == "phong" else H.SHADE_NONE,
                            camera_pos=cam["eye"], compositing=MODES[case["mode"]], gamma=0.3, iso_value=0.25)


def _network():
    """Weights of a stepping network that looks at a brick's opacity and
    spread: it skips bricks of (nearly) no opacity and steps further where the
    opacity of 32 samples (input 7) and the standard deviation (input 3) are
    small.  Layer by layer: three units, passed through the second layer."""
    w1, w2, w3 = np.zeros((16, 64), np.float32), np.zeros((64, 64), np.float32), np.zeros((64, 2), np.float32)
    for u, (f, s) in enumerate(((7, 64.0), (7, 2.0), (3, 10.0))):
        w1[f, u], w2[u, u] = s, 1.0
    w3[0, 0] = -1.0
    w3[1, 1], w3[2, 1] = -1.0, -1.0
    b3 = np.array([0.2, 2.0], np.float32)
    z = np.zeros(64, np.float32)
    return np.concatenate([w1.ravel(), z, w2.ravel(), z, w3.ravel(), b3])


def _train_inputs(case, seed):
    """Rows as the traces give them: brick statistics, TF opacities, octant; and their targets."""
    r = np.random.default_rng(seed)
    n = case["rows"]
    x = np.zeros((n, 16), np.float32)
    lo = r.random((n, 2))
    x[:, 0], x[:, 1] = lo.min(1), lo.max(1)
    x[:, 2] = x[:, 0] + (x[:, 1] - x[:, 0]) * r.random(n)
    x[:, 3] = 0.3 * (x[:, 1] - x[:, 0]) * r.random(n)
    x[:, 4] = 0.2 * r.random(n) ** 3
    x[:, 5] = 0.2 * r.random(n) ** 3
    x[:, 6] = r.random(n)
    x[:, 7] = 1 - (1 - x[:, 4]) ** 32
    x[:, 8:11] = np.where(r.random((n, 3)) < 0.5, -1.0, 1.0)
    t = np.zeros((n, 3), np.float32)
    t[:, 0] = x[:, 4] < 0.001
    t[:, 1] = np.clip(np.floor(3.5 - 12 * x[:, 3] - 4 * x[:, 4] + 0.3 * r.standard_normal(n)), 0, 3)
    t[:, 2] = np.where(t[:, 0] > 0, 0.1, 1.0)
    p = [r.uniform(-1, 1, (i, o)) * math.sqrt(6.0 / (i + o)) for i, o in ((16, 64), (64, 64), (64, 2))]
    params = np.concatenate([p[0].ravel(), np.zeros(64), p[1].ravel(), np.zeros(64), p[2].ravel(), np.zeros(2)])
    return x, t, params.astype(np.float32)


def _job_list(case, seed):
    r = _rng(seed, "jobs")
    out = []
    for j in range(case["n"]):
        dims = tuple(int(round(math.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]))))) for _ in range(3))
        out.append((dims, r.choice(["u8", "u16"]), r.randrange(1 << 30)))
    return out


def prepare(case, seed):
    ctx = _ctx()
    kind = case["kind"]
    if kind == "train":
        x, t, p = _train_inputs(case, seed)
        mlp = H.Mlp(ctx, 1)
        mlp.set_params(p)
        s = _State(case=case, mlp=mlp, close=[mlp], dx=_buffer(torch.from_numpy(x).cuda()),
                   dt=_buffer(torch.from_numpy(t).cuda()))
        torch.cuda.synchronize()
        return s
    if kind == "jobs":
        n = case["image"]
        jobs, closing, outs = [], [], []
        for dims, dtype, js in _job_list(case, seed):
            v = _device_volume(dims, dtype, "blobs", js)
            tf = ctx.transfunc(_tf(_keys("blobs", js), "u8"))
            cam = _camera(js, 3.5)
            en, ex, out = _image(n, n), _image(n, n), _image(n, n)
            torch.cuda.synchronize()
            ctx.entry_exit_device(_device_camera(cam), *_box(dims), n, n, en, ex)
            jobs.append((v, tf, en, ex, out, n, n, H.default_params(W.step_for(dims, 2.0), camera_pos=cam["eye"])))
            closing += [v, tf]
            outs.append(out.tensor)
        b = H.Batch(ctx, jobs)
        b.set_config(H.TILE_8x8, 3, 4)
        b.capture()
        return _State(case=case, batch=b, jobs=jobs, outs=outs, close=[b] + closing)
    dims, w, h = _dims(case), case["w"], case["h"]
    sp, off = _placed(dims)
    v = _device_volume(dims, case["dtype"], case["content"], seed, spacing=sp, offset=off)
    keys = _keys(case["content"], seed)
    table = _tf(keys, case["dtype"])
    tf = ctx.transfunc(table)
    cam = _camera(seed, case["radius"])
    prm = _params(case, cam)
    if kind == "host":
        first, last = _entry_exit64(cam, dims, w, h)
        s = _State(case=case, v=v, tf=tf, prm=prm, entry=first.float().cpu().numpy(), exit=last.float().cpu().numpy(),
                   out=np.zeros((h, w, 4), np.float32), close=[v, tf])
        return s
    if kind == "views":
        jobs, outs = [], []
        for k in range(case["n"]):
            c = _camera(seed, case["radius"], k, case["n"])
            en, ex, out = _image(w, h), _image(w, h), _image(w, h)
            torch.cuda.synchronize()
            ctx.entry_exit_device(_device_camera(c), *_box(dims), w, h, en, ex)
            jobs.append((v, tf, en, ex, out, w, h, _params(case, c)))
            outs.append(out.tensor)
        b = H.Batch(ctx, jobs)
        b.set_config(H.TILE_8x8, 3, 2 if case["shading"] == "phong" else 4)
        b.capture()
        return _State(case=case, batch=b, jobs=jobs, outs=outs, close=[b, v, tf])
    s = _State(case=case, v=v, tf=tf, prm=prm, keys=keys, table=table, cam=_device_camera(cam), box=_box(dims),
               en=_image(w, h), ex=_image(w, h), out=_image(w, h), close=[v, tf])
    torch.cuda.synchronize()
    if kind == "learned":
        mlp, learned = H.Mlp(ctx, 1), H.Learned(ctx, v)
        mlp.set_params(_network())
        learned.prepare(tf, prm, mlp)
        s.update(learned=learned, mlp=mlp, close=[learned, mlp, v, tf])
    elif case["classif"] == "preint" and kind == "frame":
        tf.preint_device(keys, case["table"], W.step_for(dims, case["rate"]))
    return s


def run(state):
    ctx, s = _ctx(), state
    case = s["case"]
    kind = case["kind"]
    if kind == "train":
        for _ in range(case["steps"]):
            s["mlp"].train_step_device(s["dx"], s["dt"], case["rows"], LEARNING_RATE)
        return s["mlp"].params()
    if kind in ("jobs", "views"):
        s["batch"].launch()
        return s["outs"]
    w, h = case["w"], case["h"]
    if kind == "host":
        image, stats = ctx.render(s["v"], s["tf"], s["entry"], s["exit"], s["prm"], out=s["out"])
        return [image, stats["rays"], stats["samples"]]
    ctx.entry_exit_device(s["cam"], s["box"][0], s["box"][1], w, h, s["en"], s["ex"])
    if kind == "learned":
        s["learned"].render_device(s["tf"], s["en"], s["ex"], w, h, s["prm"], s["out"])
        return s["out"].tensor
    if kind == "edit":
        old, tf = s["tf"], ctx.transfunc(s["table"])
        tf.preint_device(s["keys"], case["table"], s["prm"].step)
        s["tf"] = tf
        s["close"][1] = tf
        ctx.render_device(s["v"], tf, s["en"], s["ex"], w, h, s["prm"], s["out"])
        old.close()
        return s["out"].tensor
    ctx.render_device(s["v"], s["tf"], s["en"], s["ex"], w, h, s["prm"], s["out"])
    return s["out"].tensor


def _frame_work(dims, dtype, w, h, rate, shading, views=1):
    """Each voxel read once, each image written once; about a third of the
    rays' samples reconstructed (8 products of 4 factors, lookup,
    compositing: 60 operations), with lighting for half of those (150)."""
    voxels = dims[0] * dims[1] * dims[2]
    rays = 0.45 * w * h
    samples = rays * 0.5 * rate * max(dims) / 3.0
    return dict(bytes=voxels * (1 if dtype == "u8" else 2) + 16.0 * w * h * views,
                flops=samples * (60 + (75 if shading == "phong" else 0)) * views)


def work(case):
    kind = case["kind"]
    if kind == "train":
        per_row = 2 * (16 * 64 + 64 * 64 + 64 * 2)
        return dict(bytes=case["steps"] * case["rows"] * 76.0, flops=case["steps"] * case["rows"] * 3.0 * per_row)
    if kind == "jobs":
        mean = math.exp(0.5 * (math.log(case["lo"]) + math.log(case["hi"])))
        one = _frame_work((mean, mean, mean), "u8", case["image"], case["image"], 2.0, "none")
        return dict(bytes=case["n"] * 1.5 * one["bytes"], flops=case["n"] * 0.1 * one["flops"])
    got = _frame_work(_dims(case), case["dtype"], case["w"], case["h"], case["rate"], case["shading"],
                      case.get("n", 1))
    if kind == "host":
        got["bytes"] += 32.0 * case["w"] * case["h"]
    if case["mode"] != "dvr":   # a single value per ray is kept: no lighting of the rest
        got["flops"] = _frame_work(_dims(case), case["dtype"], case["w"], case["h"], case["rate"], "none")["flops"]
    if kind == "edit":
        got["bytes"] += 16.0 * case["table"] ** 2
        got["flops"] += 12.0 * case["table"] ** 3 / 12.0
    return got


# ---------------------------------------------------------------------------
# the same results in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _entry_exit64(cam, dims, w, h):
    """Entry and exit points of the unit-cube proxy, (h, w, 4) doubles."""
    llf, urb = (b.astype(np.float64) for b in _box(dims))
    eye, up = np.array(cam["eye"]), np.array([0.0, 1.0, 0.0])
    f = -eye / np.linalg.norm(eye)
    r = np.cross(f, up)
    r /= np.linalg.norm(r)
    u = np.cross(r, f)
    th, aspect = math.tan(math.radians(cam["fovy"]) / 2), w / h
    tu = th if aspect >= 1.0 else th / aspect
    inv = 1.0 / (urb - llf)
    dev = torch.device("cuda")
    o, fd, rd, ud = (torch.tensor(a, dtype=torch.float64, device=dev)
                     for a in ((eye - llf) * inv, f * inv, r * tu * aspect * inv, u * tu * inv))
    nx = 2 * (torch.arange(w, device=dev, dtype=torch.float64) + 0.5) / w - 1
    ny = 2 * (torch.arange(h, device=dev, dtype=torch.float64) + 0.5) / h - 1
    d = fd + nx[None, :, None] * rd + ny[:, None, None] * ud
    a, b = (0.0 - o) / d, (1.0 - o) / d
    tn = torch.minimum(a, b).amax(-1).clamp(min=cam["near"])
    tf = torch.maximum(a, b).amin(-1)
    hit = (tf > tn)[..., None]
    one = torch.ones((h, w, 1), dtype=torch.float64, device=dev)
    first = torch.cat([(o + tn[..., None] * d).clamp(0, 1), one], -1)
    last = torch.cat([(o + tf[..., None] * d).clamp(0, 1), one], -1)
    return torch.where(hit, first, 0.0), torch.where(hit, last, 0.0)


class _March64:
    def __init__(self, raw, dims, dtype, keys, step, shading="none", mode="dvr", classif="tf", filt="linear", table=0,
                 eye=(0, 0, 0)):
        self.dims, self.step, self.shading, self.mode, self.filt = dims, float(step), shading, mode, filt
        self.dev = raw.device
        self.vol = raw.reshape(-1)
        self.top = 255.0 if dtype == "u8" else 65535.0
        self.fd = torch.tensor(dims, dtype=torch.float64, device=self.dev)
        self.tf = torch.from_numpy(_tf(keys, dtype).astype(np.float64) / 255.0).to(self.dev)
        self.expo = self.step * 200.0
        self.pre = self._table(keys, table) if classif == "preint" else None
        sp, off = _placed(dims)
        self.sp, self.off, self.eye, self.light = (torch.tensor(a, dtype=torch.float64, device=self.dev)
                                                   for a in (sp, off, eye, LIGHT["pos"]))

    def _table(self, keys, n):
        """Pre-integration table [back, front]: the TF composited from front to back."""
        c8 = _lookup(keys, np.arange(n, dtype=np.float32) / np.float32(n - 1)).astype(np.float64) / 255.0
        c = torch.from_numpy(c8).to(self.dev)
        sb, sf = torch.meshgrid(torch.arange(n, device=self.dev), torch.arange(n, device=self.dev), indexing="ij")
        d, sign = (sb - sf).abs(), torch.sign(sb - sf)
        expo = self.expo / (d + 1).double()
        acc = torch.zeros((n, n, 4), dtype=torch.float64, device=self.dev)
        for j in range(n):
            s = (sf + sign * j).clamp(0, n - 1)
            live = (j <= d) & (acc[..., 3] < 0.95)
            ca = torch.where(live, 1 - (1 - c[s, 3]) ** expo, 0.0)
            wgt = ((1 - acc[..., 3]) * ca)[..., None]
            acc = acc + wgt * torch.cat([c[s, :3], torch.ones_like(wgt)], -1)
        col = acc[..., :3] / acc[..., 3:].clamp(min=0.001)
        same = torch.cat([c[:, :3], (1 - (1 - c[:, 3:]) ** self.expo)], -1)
        out = torch.cat([col, acc[..., 3:]], -1).clamp(0, 1)
        i = torch.arange(n, device=self.dev)
        out[i, i] = same
        return out

    def at(self, s):
        """Intensity at texture-space points (..., 3)."""
        m = self.fd - 1
        vp = torch.minimum((self.fd * s - 0.5).clamp(min=0.0), m)
        x, y, _ = self.dims
        if self.filt == "nearest":
            i = torch.floor(vp + 0.5).long()
            return self.vol[(i[..., 2] * y + i[..., 1]) * x + i[..., 0]].double() / self.top
        lo = torch.floor(vp)
        p = vp - lo
        lo = lo.long()
        hi = torch.minimum(lo + 1, m.long())
        total = 0.0
        for k in range(8):
            i = [hi[..., a] if k >> a & 1 else lo[..., a] for a in range(3)]
            wgt = 1.0
            for a in range(3):
                wgt = wgt * (p[..., a] if k >> a & 1 else 1 - p[..., a])
            total = total + wgt * self.vol[(i[2] * y + i[1]) * x + i[0]].double()
        return total / self.top

    def gradient(self, s):
        g = []
        for a in range(3):
            e = torch.zeros(3, dtype=torch.float64, device=self.dev)
            e[a] = 1.0 / self.dims[a]
            g.append((self.at(s - e) - self.at(s + e)) * 0.5 / self.sp[a])
        return torch.stack(g, -1)

    def phong(self, g, s, c):
        unit = torch.nn.functional.normalize
        pos = (s * self.fd - 0.5) * self.sp + self.off
        n, lv, v = unit(g, dim=-1, eps=1e-300), unit(self.light - pos, dim=-1), unit(self.eye - pos, dim=-1)
        hv = unit(v + lv, dim=-1)
        ndl = (n * lv).sum(-1, keepdim=True).clamp(min=0)
        ndh = (n * hv).sum(-1, keepdim=True).clamp(min=0)
        return (c * LIGHT["ambient"] + c * LIGHT["diffuse"] * ndl + LIGHT["specular"] * ndh ** LIGHT["shininess"])

    def border(self, first, pix, d):
        """Gradient at a ray's first sample: normal of the entry surface."""
        h, w = first.shape[:2]
        y, x = pix // w, pix % w
        unit = torch.nn.functional.normalize
        s = first[y, x, :3]
        v0 = unit(first[y, (x + 2).clamp(max=w - 1), :3] - s, dim=-1, eps=1e-300)
        v1 = unit(first[(y + 2).clamp(max=h - 1), x, :3] - s, dim=-1, eps=1e-300)
        g = torch.linalg.cross(v0, v1)
        return torch.where(((g * d).sum(-1, keepdim=True) < 0), g, -g)

    def render(self, first, last, block=8):
        h, w = first.shape[:2]
        out = torch.zeros((h * w, 4), dtype=torch.float64, device=self.dev)
        pix = (first[..., 3].reshape(-1) > 0).nonzero()[:, 0]
        o = first.reshape(-1, 4)[pix, :3]
        d = last.reshape(-1, 4)[pix, :3] - o
        end = d.norm(dim=-1)
        d = d / end[:, None]
        acc = torch.zeros((len(pix), 4), dtype=torch.float64, device=self.dev)
        best = torch.zeros(len(pix), dtype=torch.float64, device=self.dev)   # MIP / MIDA maximum
        prev = torch.zeros(len(pix), dtype=torch.float64, device=self.dev)   # previous sample (pre-integration)
        done = torch.zeros(len(pix), dtype=torch.bool, device=self.dev)
        ert = self.mode in ("dvr", "iso", "fhp", "fhn")
        k0 = 0
        while len(pix):
            t = (k0 + torch.arange(block, device=self.dev, dtype=torch.float64)) * self.step
            there = (t[None, :] <= end[:, None]) | (t == 0.0)[None, :]
            s = o[:, None, :] + t[None, :, None] * d[:, None, :]
            val = self.at(s)
            if self.pre is not None:
                n = self.pre.shape[0]
                i = torch.floor(val * (n - 1) + 0.5).long()
                j = torch.floor(torch.cat([prev[:, None], val[:, :-1]], 1) * (n - 1) + 0.5).long()
                c = self.pre[i, j]
                prev = val[:, -1]
                alpha = c[..., 3]
            else:
                c = self.tf[torch.floor(val * (len(self.tf) - 1) + 0.5).long()]
                alpha = 1 - (1 - c[..., 3]) ** self.expo if self.mode in ("dvr", "mida") else c[..., 3]
            col = c[..., :3].clone()
            hot = (there & (alpha > 0) & ~done[:, None]).nonzero()
            grad = None
            if len(hot) and (self.shading == "phong" or self.mode == "fhn"):
                a, b = hot[:, 0], hot[:, 1]
                g = self.gradient(s[a, b])
                if k0 == 0:
                    q = (b == 0).nonzero()[:, 0]
                    g[q] = self.border(first, pix[a[q]], d[a[q]])
                if self.mode == "fhn":
                    grad = torch.zeros_like(s)
                    grad[a, b] = g
                if self.shading == "phong":
                    col[a, b] = self.phong(g, s[a, b], col[a, b])
            for b in range(block):
                on = there[:, b] & ~done & (alpha[:, b] > 0)
                al, cl = alpha[:, b:b + 1], col[:, b]
                full = torch.cat([cl, al], -1)
                if self.mode == "dvr":
                    wgt = (1 - acc[:, 3:]) * al
                    new = acc + wgt * torch.cat([cl, torch.ones_like(al)], -1)
                elif self.mode == "mip":
                    up = val[:, b] > best
                    new = torch.where(up[:, None], full, acc)
                    best = torch.where(on & up, val[:, b], best)
                elif self.mode == "mop":
                    new = torch.where(al > acc[:, 3:], full, acc)
                elif self.mode == "mida":
                    gamma = 0.3
                    up = val[:, b] > best
                    mip = torch.where(up[:, None], full, acc)
                    best = torch.where(on & up, val[:, b], best)
                    # the maximum is already the sample's: no further attenuation
                    k = (1 - acc[:, 3:]) * al
                    new = gamma * mip + (1 - gamma) * (acc + k * torch.cat([cl, torch.ones_like(al)], -1))
                elif self.mode == "iso":
                    hit = (al >= 0.25 - 0.02) & (al <= 0.25 + 0.02)
                    new = torch.where(hit, torch.cat([cl, torch.ones_like(al)], -1), acc)
                else:
                    at = s[:, b] if self.mode == "fhp" else (
                        torch.nn.functional.normalize(grad[:, b], dim=-1, eps=1e-300) / 2 + 0.5
                        if grad is not None else torch.zeros_like(cl))
                    hit = (acc[:, :3] == 0).all(-1, keepdim=True)
                    new = torch.where(hit, torch.cat([at, torch.ones_like(al)], -1), acc)
                acc = torch.where(on[:, None], new, acc)
                if ert:
                    over = on & (acc[:, 3] >= 0.95)
                    acc[:, 3] = torch.where(over, 1.0, acc[:, 3])
                    done = done | over
            k0 += block
            done = done | (k0 * self.step > end)
            out[pix] = acc
            keep = (~done).nonzero()[:, 0]
            if len(keep) < 0.9 * len(pix) or not len(keep):
                pix, o, d, end, acc, best, prev, done = (v[keep] for v in (pix, o, d, end, acc, best, prev, done))
        return out.reshape(h, w, 4)


def _train64(case, seed):
    x, t, p = (torch.from_numpy(a).double().cuda() for a in _train_inputs(case, seed))
    sizes = [(16, 64), (64,), (64, 64), (64,), (64, 2), (2,)]
    parts = [v.reshape(z).clone().requires_grad_() for v, z in zip(p.split([math.prod(z) for z in sizes]), sizes)]
    mom = [[torch.zeros_like(v), torch.zeros_like(v)] for v in parts]
    gelu = torch.nn.functional.gelu
    for k in range(1, case["steps"] + 1):
        w1, b1, w2, b2, w3, b3 = parts
        y = gelu(gelu(x @ w1 + b1) @ w2 + b2) @ w3 + b3
        loss = (torch.nn.functional.binary_cross_entropy_with_logits(y[:, 0], t[:, 0], reduction="none")
                + t[:, 2] * (y[:, 1] - t[:, 1]) ** 2).mean()
        grads = torch.autograd.grad(loss, parts)
        with torch.no_grad():
            for v, g, m in zip(parts, grads, mom):
                m[0] = 0.9 * m[0] + 0.1 * g
                m[1] = 0.999 * m[1] + 0.001 * g * g
                v -= LEARNING_RATE * (m[0] / (1 - 0.9 ** k)) / ((m[1] / (1 - 0.999 ** k)).sqrt() + 1e-8)
    return torch.cat([v.detach().reshape(-1) for v in parts]).cpu()


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _train64(case, seed)
    if kind == "learned":
        return None   # a learned frame approximates the plain one: it has no value of its own in 64 bits
    if kind == "jobs":
        outs = []
        for dims, dtype, js in _job_list(case, seed):
            raw = _volume(dims, dtype, "blobs", js)
            m = _March64(raw, dims, dtype, _keys("blobs", js), _step(dims, 2.0))
            m.tf = torch.from_numpy(_tf(_keys("blobs", js), "u8").astype(np.float64) / 255.0).to(raw.device)
            outs.append(m.render(*_entry_exit64(_camera(js, 3.5), dims, case["image"], case["image"])))
        return outs
    dims = _dims(case)
    cost = 0.45 * case["w"] * case["h"] * max(dims) * case["rate"] * case.get("n", 1)
    cost *= 7 if case["shading"] == "phong" else 1
    if cost > 4.5e10:
        return None   # minutes of work in 64 bits
    raw = _volume(dims, case["dtype"], case["content"], seed)
    keys = _keys(case["content"], seed)

    def frame(cam, round_points=False):
        m = _March64(raw, dims, case["dtype"], keys, _step(dims, case["rate"]), case["shading"], case["mode"],
                     case["classif"], case["filter"], case["table"], cam["eye"])
        first, last = _entry_exit64(cam, dims, case["w"], case["h"])
        if round_points:   # the points are inputs there, in 32 bits
            first, last = first.float().double(), last.float().double()
        return m.render(first, last)

    if kind == "views":
        return [frame(_camera(seed, case["radius"], k, case["n"])) for k in range(case["n"])]
    image = frame(_camera(seed, case["radius"]), kind == "host")
    return [image, None, None] if kind == "host" else image


def _step(dims, rate):
    """The step 1 / (longest axis * rate), a float32 value."""
    return float(np.float32(1.0) / (np.float32(max(dims)) * np.float32(rate)))
