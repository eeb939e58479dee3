"""The batched launch with 2, 4 and 16 lanes per ray and every tile shape: each
job equals its single frame bit for bit.  The number of lanes follows the
launch's size, so the images are of the sizes that take each of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# image of the first job, configured batch: lanes per ray of the launch
SIZES = [((90, 70), 2, 16), ((300, 221), 2, 4), ((1301, 1201), 2, 2), ((1301, 1201), 4, 4), ((2601, 2399), 4, 2)]


@pytest.fixture(scope="module")
def volumes(ctx):
    from voreen_amd import hipdvr as H, workloads as W
    out = []
    for seed, dims, dtype in ((3, (96, 80, 72), H.U16), (5, (40, 56, 33), H.U8)):
        v = ctx.volume(H.synth_blobs(seed, dims, dtype))
        t = ctx.transfunc(H.tf_from_keys(W.random_keys(seed + 4, 5), 256 if dtype == H.U8 else 4096))
        out.append((v, t, dims))
    yield out
    for v, t, _ in out:
        v.close()
        t.close()


@pytest.mark.parametrize("image,batch,lanes", SIZES, ids=[f"{s[0][0]}x{s[0][1]}-{s[2]}lanes" for s in SIZES])
@pytest.mark.parametrize("shading", [0, 1])
def test_every_lane_count_and_tile_shape(ctx, volumes, image, batch, lanes, shading):
    from voreen_amd import hipdvr as H, workloads as W
    jobs, refs = [], []
    # a second, small and ragged job of the other voxel type, its rays shorter
    for (v, t, dims), (w, h) in zip(volumes, (image, (37, 19))):
        de, dx, do = (ctx.alloc(w * h * 16) for _ in range(3))
        llf, urb = W.world_box(dims)
        cam = W.orbit_camera(7, 36, radius=2.3)
        ctx.entry_exit_device(cam, llf, urb, w, h, de, dx)
        p = H.default_params(W.step_for(dims, 2.0), shading=shading, camera_pos=tuple(cam.eye))
        ctx.render_device(v, t, de, dx, w, h, p, do)
        ctx.synchronize()
        refs.append(do.download((h, w, 4), np.float32))
        jobs.append((v, t, de, dx, do, w, h, p))
    assert np.mean(refs[0][..., 3] > 0) > 0.05
    b = H.Batch(ctx, jobs)
    try:
        for tile in (0, 1, 2):
            print(f"[case] batch {image} {lanes} lanes tile {tile} shading {shading}", flush=True)
            b.set_config(tile, 3, batch)
            for j, r in zip(jobs, refs):
                j[4].upload(np.full(r.shape, -1.0, np.float32))
            b.launch()
            ctx.synchronize()
            for i, (j, r) in enumerate(zip(jobs, refs)):
                assert np.array_equal(j[4].download(r.shape, np.float32), r), f"job {i} tile {tile}"
    finally:
        b.close()
        for j in jobs:
            for x in j[2:5]:
                x.free()
