"""The frame march with 2, 4 and 16 lanes per ray, its skip grid and its tile
order against the reference-layout kernel (no skipping, one lane per ray): the
same floats in the same order, so the images and sample counts are equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def sparse_volume(seed, dims, dtype, fill):
    """Mostly zero voxels with a few random ones: every distance of the skip
    grid, bricks cut by the volume's edge, single occupied voxels at corners."""
    r = np.random.default_rng(seed)
    x, y, z = dims
    top = 255 if dtype == np.uint8 else 65535
    v = np.zeros((z, y, x), dtype)
    n = max(1, int(fill * v.size))
    at = r.integers(0, v.size, n)
    v.reshape(-1)[at] = r.integers(1, top + 1, n)
    v[0, 0, 0] = v[-1, -1, -1] = top
    return v


CASES = [
    # dims, dtype, image, fill, loop cap
    ((1, 1, 1), np.uint8, (3, 2), 1.0, 0),
    ((2, 9, 8), np.uint16, (17, 33), 0.2, 0),
    ((7, 65, 130), np.uint8, (64, 48), 1e-3, 0),
    ((257, 33, 16), np.uint16, (129, 65), 2e-4, 0),
    ((140, 150, 129), np.uint16, (300, 140), 3e-6, 0),
    ((96, 96, 96), np.uint8, (1, 1), 1e-3, 0),
    ((96, 80, 72), np.uint16, (90, 70), 1e-2, 1),
    ((96, 80, 72), np.uint16, (90, 70), 1e-2, 37),
]


@pytest.mark.parametrize("dims,dtype,image,fill,cap", CASES, ids=[f"{c[0]}-{c[2]}-cap{c[4]}" for c in CASES])
@pytest.mark.parametrize("shading,exact", [(0, 0), (1, 1)])
def test_lanes_equal_the_reference_kernel(ctx, dims, dtype, image, fill, cap, shading, exact):
    from voreen_amd import hipdvr as H, workloads as W
    print(f"[case] lanes {dims} {np.dtype(dtype).name} {image} cap {cap} shading {shading}", flush=True)
    v = ctx.volume(sparse_volume(sum(dims), dims, dtype, fill))
    # alpha 0 at the low end: zero voxels are empty space
    t = ctx.transfunc(H.tf_from_keys([(0.0, (9, 200, 30, 0)), (0.05, (9, 200, 30, 0)), (0.3, (200, 10, 90, 60)),
                                      (1.0, (255, 255, 0, 200))], 256))
    w, h = image
    de, dx, do = (ctx.alloc(w * h * 16) for _ in range(3))
    try:
        llf, urb = W.world_box(dims)
        cam = W.orbit_camera(5, 36, radius=1.9)
        ctx.entry_exit_device(cam, llf, urb, w, h, de, dx)
        out = {}
        for lanes, kernel, batch in (("ref", H.KERNEL_REFERENCE, 0), ("auto", H.KERNEL_CELL, 0),
                                     (2, H.KERNEL_CELL, 2), (4, H.KERNEL_CELL, 4), (16, H.KERNEL_CELL, 8)):
            p = H.default_params(W.step_for(dims, 2.0), shading=shading, exact_shading=exact, kernel=kernel,
                                 batch=batch, camera_pos=tuple(cam.eye))
            p.loop_cap = cap
            do.upload(np.full((h, w, 4), np.nan, np.float32))
            st = ctx.render_device(v, t, de, dx, w, h, p, do, stats=True)
            out[lanes] = (do.download((h, w, 4), np.float32), st)
            assert not np.isnan(out[lanes][0]).any(), f"{lanes}: pixel not written"
        ref, rs = out["ref"]
        for lanes in ("auto", 2, 4, 16):
            img, st = out[lanes]
            assert np.array_equal(img, ref), f"{lanes} lanes"
            assert (st["samples"], st["shaded"], st["rays"]) == (rs["samples"], rs["shaded"], rs["rays"]), f"{lanes}"
    finally:
        for b in (de, dx, do):
            b.free()
        v.close()
        t.close()
