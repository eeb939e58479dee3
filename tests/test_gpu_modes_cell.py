"""The compositing modes and the pre-integrated classification on the cell
records (several lanes per ray, samples skipped that cannot contribute)
against the reference-layout kernels, which take every sample: the same floats
in the same order, so images and counters of samples are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = [(0.0, (9, 200, 30, 0)), (0.12, (9, 200, 30, 0)), (0.3, (200, 10, 90, 60)), (0.45, (20, 250, 90, 0)),
        (0.6, (20, 250, 90, 0)), (1.0, (255, 255, 0, 200))]

# dims, dtype, image, loop cap, lanes (hipdvr_params::batch)
SHAPES = [
    ((1, 1, 1), np.uint8, (3, 2), 0, 0),
    ((2, 9, 8), np.uint16, (17, 33), 0, 0),
    ((7, 65, 130), np.uint8, (64, 48), 0, 4),
    ((129, 33, 16), np.uint16, (129, 65), 0, 8),
    ((96, 80, 72), np.uint16, (90, 70), 1, 0),
    ((96, 80, 72), np.uint8, (90, 70), 37, 4),
    ((72, 80, 96), np.uint16, (160, 130), 0, 8),
]


def volume(dims, dtype):
    """Zero space, a smooth blob and scattered single voxels."""
    x, y, z = dims
    top = 255 if dtype == np.uint8 else 65535
    g = np.meshgrid(*(np.linspace(-1, 1, n) if n > 1 else np.zeros(1) for n in (z, y, x)), indexing="ij")
    r2 = g[0] ** 2 + g[1] ** 2 + g[2] ** 2
    v = np.clip(1.0 - 2.2 * r2, 0.0, 0.8)
    r = np.random.default_rng(x + y + z)
    v.reshape(-1)[r.integers(0, v.size, max(1, v.size // 4000))] = r.random(max(1, v.size // 4000))
    v[0, 0, 0] = 1.0
    return (v * top).astype(dtype)


class Scene:
    def __init__(self, ctx, dims, dtype, image, cap, lanes):
        from voreen_amd import hipdvr as H, workloads as W
        self.ctx, self.H, self.W = ctx, H, W
        self.dims, self.image, self.cap, self.lanes = dims, image, cap, lanes
        self.vol = ctx.volume(volume(dims, dtype))
        self.tf = ctx.transfunc(H.tf_from_keys(KEYS, 256))
        self.bufs = [ctx.alloc(image[0] * image[1] * 16) for _ in range(3)]
        llf, urb = W.world_box(dims)
        self.cam = W.orbit_camera(5, 36, radius=1.9)
        ctx.entry_exit_device(self.cam, llf, urb, *image, self.bufs[0], self.bufs[1])

    def close(self):
        for b in self.bufs:
            b.free()
        self.vol.close()
        self.tf.close()

    def frame(self, kernel, stats, step=None, **params):
        de, dx, do = self.bufs
        w, h = self.image
        p = self.H.default_params(step or self.W.step_for(self.dims, 2.0), kernel=kernel, batch=self.lanes,
                                  camera_pos=tuple(self.cam.eye), **params)
        p.loop_cap = self.cap
        do.upload(np.full((h, w, 4), np.nan, np.float32))
        st = self.ctx.render_device(self.vol, self.tf, de, dx, w, h, p, do, stats=stats)
        return do.download((h, w, 4), np.float32), st

    def compare(self, what, **kw):
        print(f"[case] modes cell {self.dims} {self.image} cap {self.cap} {what}", flush=True)
        ref, rs = self.frame(self.H.KERNEL_REFERENCE, True, **kw)
        img, st = self.frame(self.H.KERNEL_AUTO, True, **kw)
        quiet, _ = self.frame(self.H.KERNEL_AUTO, False, **kw)
        assert np.array_equal(img, ref), what
        assert np.array_equal(quiet, ref), f"{what} without counters"
        assert (st["rays"], st["samples"], st["shaded"]) == (rs["rays"], rs["samples"], rs["shaded"]), what
        assert st["fetched"] <= rs["fetched"] + 16 * rs["rays"], what   # a run's last sample may be read twice


@pytest.mark.parametrize("dims,dtype,image,cap,lanes", SHAPES, ids=[f"{s[0]}-{s[2]}-cap{s[3]}" for s in SHAPES])
@pytest.mark.parametrize("shading", [0, 1])
def test_modes_equal_the_reference_kernel(ctx, dims, dtype, image, cap, lanes, shading):
    s = Scene(ctx, dims, dtype, image, cap, lanes)
    H = s.H
    try:
        for mode in (H.COMPOSITE_MIP, H.COMPOSITE_MOP, H.COMPOSITE_MIDA, H.COMPOSITE_ISO, H.COMPOSITE_FHP,
                     H.COMPOSITE_FHN):
            for gamma in ((0.0, 0.4) if mode == H.COMPOSITE_MIDA else (0.0,)):
                for iso in ((0.1, 0.25, 0.9) if mode == H.COMPOSITE_ISO else (0.5,)):
                    s.compare(f"mode {mode} gamma {gamma} iso {iso} shading {shading}", compositing=mode, gamma=gamma,
                              iso_value=iso, shading=shading)
    finally:
        s.close()


def tables(H, step):
    yield "small", H.preint_build(KEYS, 2, step)
    yield "keys", H.preint_build(KEYS, 256, step)
    yield "integral", H.preint_build(KEYS, 100, step, use_integral=True)
    r = np.random.default_rng(3)
    t = np.zeros((300, 300, 4), np.float32)   # visible only where a low and a high index meet
    t[:60, 150:] = r.random((60, 150, 4))
    t[200:, 20:40] = r.random((100, 20, 4))
    yield "jumps", t
    yield "nothing", np.zeros((64, 64, 4), np.float32)


@pytest.mark.parametrize("dims,dtype,image,cap,lanes", SHAPES, ids=[f"{s[0]}-{s[2]}-cap{s[3]}" for s in SHAPES])
@pytest.mark.parametrize("shading", [0, 1])
def test_preint_equals_the_reference_kernel(ctx, dims, dtype, image, cap, lanes, shading):
    s = Scene(ctx, dims, dtype, image, cap, lanes)
    try:
        step = s.W.step_for(dims, 2.0)
        for name, table in tables(s.H, step):
            s.tf.set_preint(np.ascontiguousarray(table, np.float32))
            # samples half a voxel apart, five, and more than a brick of the skip grid
            for st in (step, 5.0 / max(dims), 11.0 / max(dims)):
                s.compare(f"preint {name} step {st:.4f} shading {shading}", step=st, classification=s.H.CLASS_PREINT,
                          shading=shading)
    finally:
        s.close()
