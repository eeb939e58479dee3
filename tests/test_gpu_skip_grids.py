"""Skip grids of the cell kernels where several frames hold them: a captured
frame between frames of other modes and transfer functions, and frames of one
volume on several streams without a wait between them.  Every image is the one
the reference-layout kernel (no skip grid) gives."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = [(0.0, (9, 200, 30, 0)), (0.12, (9, 200, 30, 0)), (0.3, (200, 10, 90, 60)), (0.45, (20, 250, 90, 0)),
        (0.6, (20, 250, 90, 0)), (1.0, (255, 255, 0, 200))]
OTHER = [(0.0, (200, 20, 30, 0)), (0.7, (200, 20, 30, 0)), (0.75, (90, 10, 90, 250)), (1.0, (25, 255, 0, 90))]


class Runtime:
    """Streams and graphs of the HIP runtime that the library is linked to."""

    def __init__(self):
        from voreen_amd import hipdvr as H
        H.load()
        path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line)
        self.lib = C.CDLL(path)

    def call(self, name, *args):
        rc = getattr(self.lib, name)(*args)
        assert rc == 0, f"{name}: {rc}"

    def stream(self):
        s = C.c_void_p()
        self.call("hipStreamCreateWithFlags", C.byref(s), 1)
        return s

    def capture(self, stream, body):
        """An executable graph of what body submits to the stream (global mode)."""
        graph, run = C.c_void_p(), C.c_void_p()
        self.call("hipStreamBeginCapture", stream, 0)
        try:
            body()
        finally:
            self.call("hipStreamEndCapture", stream, C.byref(graph))
        self.call("hipGraphInstantiate", C.byref(run), graph, None, None, C.c_size_t(0))
        self.call("hipGraphDestroy", graph)
        return run

    def replay(self, run, stream):
        self.call("hipGraphLaunch", run, stream)
        self.call("hipStreamSynchronize", stream)


def volume(dims):
    x, y, z = dims
    g = np.meshgrid(*(np.linspace(-1, 1, n) for n in (z, y, x)), indexing="ij")
    return (np.clip(1.0 - 1.7 * (g[0] ** 2 + g[1] ** 2 + g[2] ** 2), 0.0, 1.0) * 65535).astype(np.uint16)


class Scene:
    """One volume, two TFs, a frame of every kind that has a skip rule."""

    def __init__(self, dims, image):
        from voreen_amd import hipdvr as H, workloads as W
        self.H, self.dims, self.image = H, dims, image
        self.ctx = H.Context(0)
        self.vol = self.ctx.volume(volume(dims))
        self.step = W.step_for(dims, 2.0)
        self.tfs = [self.ctx.transfunc(H.tf_from_keys(k, 256)) for k in (KEYS, OTHER)]
        for t, k in zip(self.tfs, (KEYS, OTHER)):
            t.set_preint(np.ascontiguousarray(H.preint_build(k, 128, self.step), np.float32))
        self.de, self.dx, self.do, self.dg = (self.ctx.alloc(image[0] * image[1] * 16) for _ in range(4))
        llf, urb = W.world_box(dims)
        self.ctx.entry_exit_device(W.orbit_camera(5, 36, radius=1.9), llf, urb, *image, self.de, self.dx)
        self.ctx.synchronize()
        self.kinds = {"dvr": {}, "mip": dict(compositing=H.COMPOSITE_MIP),
                      "iso": dict(compositing=H.COMPOSITE_ISO, iso_value=0.2),
                      "preint": dict(classification=H.CLASS_PREINT)}
        self.ref = {(k, t): self.frame(k, t, H.KERNEL_REFERENCE) for k in self.kinds for t in (0, 1)}
        for a in self.kinds:   # the frames differ, or a wrong grid would show nothing
            for b in self.kinds:
                assert a == b or not np.array_equal(self.ref[a, 0], self.ref[b, 0])

    def stream(self, s):
        self.ctx.check(self.ctx.lib.hipdvr_set_stream(self.ctx.h, s), "hipdvr_set_stream")

    def render(self, kind, tf, kernel=0, out=None):
        w, h = self.image
        p = self.H.default_params(self.step, kernel=kernel, **self.kinds[kind])
        self.ctx.render_device(self.vol, self.tfs[tf], self.de, self.dx, w, h, p, out or self.do)

    def image_of(self, buf):
        self.ctx.synchronize()
        return buf.download((self.image[1], self.image[0], 4), np.float32)

    def frame(self, kind, tf, kernel=0):
        self.render(kind, tf, kernel)
        return self.image_of(self.do)

    def check(self, kind, tf, what):
        assert np.array_equal(self.frame(kind, tf), self.ref[kind, tf]), f"{what}: {kind} of TF {tf}"

    def close(self):
        self.stream(None)
        for b in (self.de, self.dx, self.do, self.dg):
            b.free()
        for o in (self.vol, *self.tfs):
            o.close()
        self.ctx.close()


@pytest.fixture()
def scene():
    s = Scene((120, 96, 88), (150, 130))
    yield s
    s.close()


@pytest.mark.parametrize("warm", [True, False], ids=["built-before", "built-in-graph"])
def test_captured_frame_between_other_frames(scene, warm):
    s, rt = scene, Runtime()
    print(f"[case] skip grids: captured DVR frame, grid {'built before' if warm else 'built in the graph'}", flush=True)
    s.check("dvr", 0 if warm else 1, "before the capture")   # the cell records, and TF 0's grid if warm
    side = rt.stream()
    s.stream(side)
    g = rt.capture(side, lambda: s.render("dvr", 0, out=s.dg))
    if not warm:
        s.check("dvr", 0, "eager, before the first replay")
    for rep, (kind, tf) in enumerate([("iso", 0), ("preint", 0), ("dvr", 1), ("iso", 1), ("mip", 0), ("dvr", 0)]):
        s.check(kind, tf, f"round {rep}")
        s.dg.upload(np.full((s.image[1], s.image[0], 4), -1.0, np.float32))
        rt.replay(g, side)
        assert np.array_equal(s.image_of(s.dg), s.ref["dvr", 0]), f"replay {rep} after {kind} of TF {tf}"
    # a second graph of another mapping beside the first
    g2 = rt.capture(side, lambda: s.render("dvr", 1, out=s.dg))
    for rep in range(3):
        rt.replay(g, side)
        assert np.array_equal(s.image_of(s.dg), s.ref["dvr", 0]), f"first graph, {rep}"
        rt.replay(g2, side)
        assert np.array_equal(s.image_of(s.dg), s.ref["dvr", 1]), f"second graph, {rep}"
        s.check("iso", rep % 2, f"between, {rep}")
    for x in (g, g2):
        rt.call("hipGraphExecDestroy", x)
    s.stream(None)
    rt.call("hipStreamDestroy", side)


def test_frames_on_several_streams(scene):
    s, rt = scene, Runtime()
    print("[case] skip grids: frames of one volume on three streams", flush=True)
    s.check("dvr", 0, "the cell records")
    streams = [rt.stream() for _ in range(3)]
    w, h = s.image
    work = [(k, t) for t in (0, 1, 0) for k in ("dvr", "iso", "mip", "preint", "dvr", "preint", "iso", "mip")]
    outs = [s.ctx.alloc(w * h * 16) for _ in work]
    try:
        for i, (kind, tf) in enumerate(work):
            s.stream(streams[i % 3])
            s.render(kind, tf, out=outs[i])
        for st in streams:
            rt.call("hipStreamSynchronize", st)
        for (kind, tf), o in zip(work, outs):
            assert np.array_equal(s.image_of(o), s.ref[kind, tf]), f"{kind} of TF {tf}"
    finally:
        for o in outs:
            o.free()
        s.stream(None)
        for st in streams:
            rt.call("hipStreamDestroy", st)
