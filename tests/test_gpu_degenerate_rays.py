"""Rays whose entry or exit point is not a number: all their samples take the
TF's first entry, whatever the skip grid says about the brick at the origin
(which the clamps map them to).  Every kernel gives the reference-layout
kernel's image."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first_visible", [True, False])
@pytest.mark.parametrize("cap", [1, 5, 37])
def test_degenerate_rays_equal_the_reference_kernel(ctx, first_visible, cap):
    from voreen_amd import hipdvr as H
    w, h, n = 24, 20, 32
    # the first entries visible or not; the 8^3 brick at the origin invisible,
    # its neighbours visible
    a0 = 90 if first_visible else 0
    keys = [(0.0, (9, 200, 30, a0)), (0.1, (9, 200, 30, a0)), (0.12, (9, 200, 30, 0)), (0.5, (9, 20, 130, 0)),
            (0.52, (200, 10, 90, 60)), (0.8, (200, 10, 90, 60)), (0.82, (20, 250, 90, 0)), (1.0, (20, 250, 90, 0))]
    vol = np.full((n, n, n), 150, np.uint8)
    vol[:10, :10, :10] = 240
    v, t = ctx.volume(vol), ctx.transfunc(H.tf_from_keys(keys, 256))
    r = np.random.default_rng(4)
    en = np.ones((h, w, 4), np.float32)
    en[..., :3] = r.random((h, w, 3))
    ex = np.ones((h, w, 4), np.float32)
    ex[..., :3] = r.random((h, w, 3))
    for img, pick in ((en, r.random((h, w, 3)) < 0.1), (ex, r.random((h, w, 3)) < 0.1)):
        img[..., :3][pick] = np.nan
    ex[0, :, 0] = np.inf
    de, dx, do = (ctx.alloc(w * h * 16) for _ in range(3))
    try:
        de.upload(en)
        dx.upload(ex)

        def frame(kernel, batch):
            p = H.default_params(1.0 / 64, kernel=kernel, batch=batch)
            p.loop_cap = cap
            st = ctx.render_device(v, t, de, dx, w, h, p, do, stats=True)
            return do.download((h, w, 4), np.float32), st, p

        ref, rs, p = frame(H.KERNEL_REFERENCE, 0)
        for batch in (0, 2, 4, 8):
            print(f"[case] degenerate rays, first entry {a0}, cap {cap}, batch {batch}", flush=True)
            img, st, _ = frame(H.KERNEL_CELL, batch)
            assert np.array_equal(img, ref), f"batch {batch}"
            assert (st["samples"], st["rays"]) == (rs["samples"], rs["rays"]), f"batch {batch}"
        b = H.Batch(ctx, [(v, t, de, dx, do, w, h, p)])
        try:
            b.set_config(0, 3, 2)
            b.launch()
            ctx.synchronize()
            assert np.array_equal(do.download((h, w, 4), np.float32), ref), "batched"
        finally:
            b.close()
    finally:
        for x in (de, dx, do):
            x.free()
        v.close()
        t.close()
