"""The learned march with 1, 2 and 4 lanes per ray: its samples do not depend
on the number of lanes, whatever the loop cap, so a frame of 2 lanes, one of 4 and the batched
launch (by its size 4 lanes, 2, or one with several samples in flight) give the
same image bit for bit, and a frame large enough for one lane the image that 2
lanes give."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def network(H, ctx):
    """Skips nearly transparent bricks, steps further where the opacity of 32
    samples (input 7) and the standard deviation (input 3) are small."""
    w1, w2, w3 = np.zeros((16, 64), np.float32), np.zeros((64, 64), np.float32), np.zeros((64, 2), np.float32)
    for u, (f, s) in enumerate(((7, 64.0), (7, 2.0), (3, 10.0))):
        w1[f, u], w2[u, u] = s, 1.0
    w3[0, 0], w3[1, 1], w3[2, 1] = -1.0, -1.0, -1.0
    z = np.zeros(64, np.float32)
    m = H.Mlp(ctx)
    m.set_params(np.concatenate([w1.ravel(), z, w2.ravel(), z, w3.ravel(), np.array([0.2, 2.0], np.float32)]))
    return m


class Scene:
    def __init__(self, ctx, dims, dtype):
        from voreen_amd import hipdvr as H, workloads as W
        self.ctx, self.H, self.W, self.dims = ctx, H, W, dims
        vol = W.make_volume("c1", dims=dims)
        self.vol = ctx.volume((vol >> 8).astype(np.uint8) if dtype == np.uint8 else vol)
        keys, _ = W.make_tf("c1")
        self.tf = ctx.transfunc(H.tf_from_keys(keys, 4096))
        self.net = network(H, ctx)
        self.learned = H.Learned(ctx, self.vol)
        self.opts = H.learned_opts(psnr_floor=1e-3)   # the judge accepts everything

    def view(self, image, cap, shading, radius=2.1):
        w, h = image
        de, dx, do = (self.ctx.alloc(w * h * 16) for _ in range(3))
        llf, urb = self.W.world_box(self.dims)
        cam = self.W.orbit_camera(5, 36, radius=radius)
        self.ctx.entry_exit_device(cam, llf, urb, w, h, de, dx)
        p = self.H.default_params(self.W.step_for(self.dims, 2.0), shading=shading, camera_pos=tuple(cam.eye))
        p.loop_cap = cap
        return de, dx, do, p

    def frame(self, bufs, image, batch):
        de, dx, do, p = bufs
        p.batch = batch
        do.upload(np.full((image[1], image[0], 4), -1.0, np.float32))
        st = self.learned.render_device(self.tf, de, dx, image[0], image[1], p, do, opts=self.opts, stats=True)
        assert not st["fell_back"]
        return do.download((image[1], image[0], 4), np.float32)

    def close(self):
        for o in (self.learned, self.net, self.vol, self.tf):
            o.close()


@pytest.mark.parametrize("dims,dtype,image", [((96, 80, 72), np.uint16, (90, 70)), ((130, 65, 33), np.uint8, (64, 129))],
                         ids=["u16", "u8"])
@pytest.mark.parametrize("shading", [0, 1])
def test_samples_do_not_depend_on_the_lanes(ctx, dims, dtype, image, shading):
    s = Scene(ctx, dims, dtype)
    H = s.H
    try:
        for cap in (0, 1, 2, 3, 5, 6, 37, 150):
            print(f"[case] learned lanes {dims} {image} shading {shading} cap {cap}", flush=True)
            bufs = s.view(image, cap, shading)
            de, dx, do, p = bufs
            s.learned.prepare(s.tf, p, s.net, opts=s.opts)
            two, four = s.frame(bufs, image, 2), s.frame(bufs, image, 4)
            b = H.Batch(ctx, [(s.vol, s.tf, de, dx, do, image[0], image[1], p)])
            try:
                b.set_learned([s.learned], s.opts)
                for tile in (0, 1, 2):
                    b.set_config(tile, 4, 2)
                    do.upload(np.full((image[1], image[0], 4), -1.0, np.float32))
                    b.launch_learned(stats=True)
                    one = do.download((image[1], image[0], 4), np.float32)
                    assert np.array_equal(two, one), f"cap {cap} tile {tile}: 2 lanes"
                    assert np.array_equal(four, one), f"cap {cap} tile {tile}: 4 lanes"
                assert cap or np.mean(one[..., 3] > 0) > 0.1
            finally:
                b.close()
            for x in (de, dx, do):
                x.free()
    finally:
        s.close()


@pytest.mark.parametrize("shading,image", [(0, (1001, 819)), (1, (1331, 997))])
def test_large_frame_equals_two_lanes(ctx, shading, image):
    s = Scene(ctx, (64, 72, 80), np.uint16)
    try:
        print(f"[case] learned one lane {image} shading {shading}", flush=True)
        bufs = s.view(image, 0, shading)
        s.learned.prepare(s.tf, bufs[3], s.net, opts=s.opts)
        assert np.array_equal(s.frame(bufs, image, 0), s.frame(bufs, image, 2))
        for x in bufs[:3]:
            x.free()
    finally:
        s.close()


# pixels of the first image: two lanes per ray, one (unshaded, with Phong)
@pytest.mark.parametrize("shading,image", [(0, (1301, 1201)), (1, (1301, 1201)), (0, (3103, 2917)), (1, (3607, 3391))],
                         ids=["unshaded-2", "phong-2", "unshaded-1", "phong-1"])
def test_large_batch_equals_two_lane_frames(ctx, shading, image):
    """Learned views of both voxel types and odd sizes and a plain one, in a
    launch of 1.5 to 6 M pixels and in one large enough for one lane."""
    scenes = [Scene(ctx, (64, 72, 80), np.uint16), Scene(ctx, (60, 48, 52), np.uint8)]
    jobs = [(scenes[i], im) for i, im in ((0, image), (1, (131, 57)), (0, (40, 37)), (1, (63, 129)))]
    plain = 2
    views = [(s, im, s.view(im, 0, shading)) for s, im in jobs]
    try:
        print(f"[case] learned batch {image} shading {shading}", flush=True)
        for s in scenes:
            s.learned.prepare(s.tf, next(v[2][3] for v in views if v[0] is s), s.net, opts=s.opts)
        ref = []
        for i, (s, im, bufs) in enumerate(views):
            if i != plain:
                ref.append(s.frame(bufs, im, 2))
                continue
            de, dx, do, p = bufs
            s.ctx.render_device(s.vol, s.tf, de, dx, im[0], im[1], p, do)
            s.ctx.synchronize()
            ref.append(do.download((im[1], im[0], 4), np.float32))
        b = scenes[0].H.Batch(ctx, [(s.vol, s.tf, de, dx, do, im[0], im[1], p) for s, im, (de, dx, do, p) in views])
        try:
            b.set_learned([None if i == plain else v[0].learned for i, v in enumerate(views)], scenes[0].opts)
            for tile, resident in ((0, 0), (1, 2), (2, 8)):
                b.set_config(tile, 3, 2, resident)
                for v, r in zip(views, ref):
                    v[2][2].upload(np.full(r.shape, -1.0, np.float32))
                b.launch_learned(stats=True)
                for i, (v, r) in enumerate(zip(views, ref)):
                    assert np.array_equal(v[2][2].download(r.shape, np.float32), r), f"view {i} tile {tile}"
        finally:
            b.close()
        for v in views:
            for x in v[2][:3]:
                x.free()
    finally:
        for s in scenes:
            s.close()


@pytest.mark.parametrize("shading", [0, 1])
def test_records_past_4_gib(ctx, shading):
    """Volumes addressed with 64 bits: batches of 4 and 2 lanes and a frame
    large enough for one lane elsewhere, against frames of 2 and 4 lanes."""
    from voreen_amd import hipdvr as H, workloads as W
    s = Scene.__new__(Scene)
    s.ctx, s.H, s.W, s.dims = ctx, H, W, (2048, 1024, 144)
    vox, _ = ctx.synth_turbulence(0x51, s.dims, 0.4)
    s.vol = ctx.volume_device(vox, s.dims, H.U16)
    vox.free()
    _, tf = W.make_tf("c4")
    s.tf, s.net = ctx.transfunc(tf), network(H, ctx)
    s.learned, s.opts = H.Learned(ctx, s.vol), H.learned_opts(psnr_floor=1e-3)
    try:
        for image in ((131, 77), (1381, 1301)):
            print(f"[case] learned 64-bit {image} shading {shading}", flush=True)
            bufs = s.view(image, 0, shading, radius=1.4)
            de, dx, do, p = bufs
            s.learned.prepare(s.tf, p, s.net, opts=s.opts)
            two, four = s.frame(bufs, image, 2), s.frame(bufs, image, 4)
            assert np.mean(two[..., 3] > 0) > 0.1
            assert np.array_equal(two, four) and np.array_equal(two, s.frame(bufs, image, 0))
            b = H.Batch(ctx, [(s.vol, s.tf, de, dx, do, image[0], image[1], p)])
            try:
                b.set_learned([s.learned], s.opts)
                b.set_config(0, 3, 2)
                do.upload(np.full(two.shape, -1.0, np.float32))
                b.launch_learned(stats=True)
                assert np.array_equal(two, do.download(two.shape, np.float32))
            finally:
                b.close()
            for x in (de, dx, do):
                x.free()
    finally:
        s.close()


@pytest.mark.parametrize("shading,exact", [(0, 0), (1, 0), (1, 1)])
def test_judge_pixels_equal_the_plain_frame(ctx, shading, exact):
    s = Scene(ctx, (96, 80, 72), np.uint16)
    H, image = s.H, (200, 170)
    try:
        print(f"[case] judge pixels shading {shading} exact {exact}", flush=True)
        de, dx, do, p = bufs = s.view(image, 0, shading)
        p.exact_shading = exact
        s.ctx.render_device(s.vol, s.tf, de, dx, image[0], image[1], p, do)
        s.ctx.synchronize()
        plain = do.download((image[1], image[0], 4), np.float32)
        gw, gh = H.learned_sparse_dims(*image)
        ds = ctx.alloc(gw * gh * 16)
        assert s.learned.sparse_remarch(s.tf, de, dx, image[0], image[1], p, ds) == (gw, gh)
        xs, ys = ([(g // 8) * 64 + 28 + g % 8 for g in range(n)] for n in (gw, gh))
        assert np.array_equal(ds.download((gh, gw, 4), np.float32), plain[np.ix_(ys, xs)])
        for x in (*bufs[:3], ds):
            x.free()
    finally:
        s.close()


@pytest.mark.parametrize("images", [[(700, 600), (40, 37), (130, 57)], [(40, 37)] * 260], ids=["uneven", "many"])
@pytest.mark.parametrize("shading", [0, 1])
def test_fallback_frames_equal_the_plain_frames(ctx, shading, images):
    """The views of a batch fall back (uint8 and uint16 volumes, uneven images,
    many views), then every second one."""
    scenes = [Scene(ctx, (64, 72, 80), np.uint16), Scene(ctx, (60, 48, 52), np.uint8)]
    H = scenes[0].H
    bad = H.Mlp(ctx, seed=3)
    w = bad.params()
    w[-2] = 50.0      # skip every brick
    bad.set_params(w)
    views, bufs = [], {}
    for i, image in enumerate(images):
        key = (i % 2, image)
        if key not in bufs:
            bufs[key] = scenes[i % 2].view(image, 0, shading, radius=1.0)   # (judge pixels see the volume)
        de, dx, _, p = bufs[key]
        views.append((scenes[i % 2], de, dx, ctx.alloc(image[0] * image[1] * 16), image, p))
    try:
        print(f"[case] learned fallback {len(images)} views shading {shading}", flush=True)
        ref = []
        for s, de, dx, do, image, p in views:
            s.ctx.render_device(s.vol, s.tf, de, dx, image[0], image[1], p, do)
            s.ctx.synchronize()
            ref.append(do.download((image[1], image[0], 4), np.float32))
        for s in scenes:
            s.learned.prepare(s.tf, next(v[5] for v in views if v[0] is s), bad)
        b = H.Batch(ctx, [(s.vol, s.tf, de, dx, do, image[0], image[1], p) for s, de, dx, do, image, p in views])
        try:
            for step in (1, 2):
                b.set_learned([v[0].learned if i % step == 0 else None for i, v in enumerate(views)])
                for v, r in zip(views, ref):
                    v[3].upload(np.full(r.shape, -1.0, np.float32))
                st = b.launch_learned(stats=True)
                for i, (v, r) in enumerate(zip(views, ref)):
                    assert st[i]["fell_back"] == (i % step == 0), f"view {i} of every {step}"
                    assert np.array_equal(v[3].download(r.shape, np.float32), r), f"view {i} of every {step}"
        finally:
            b.close()
    finally:
        for v in views:
            v[3].free()
        for de, dx, do, _ in bufs.values():
            for x in (de, dx, do):
                x.free()
        bad.close()
        for s in scenes:
            s.close()
