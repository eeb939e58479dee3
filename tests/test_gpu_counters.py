"""Frame statistics beyond 32 bits: rays of 2^27 samples each, whose sum over
one wavefront passes 2^32."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_sums_of_a_wavefront_have_64_bits(ctx):
    from voreen_amd import hipdvr as H
    w = h = 8
    cap = 1 << 27
    v = ctx.volume(np.zeros((16, 16, 16), np.uint8))
    t = ctx.transfunc(H.tf_from_keys([(0.0, (9, 200, 30, 0)), (0.05, (9, 200, 30, 0)), (1.0, (255, 255, 0, 200))], 256))
    de, dx, do = (ctx.alloc(w * h * 16) for _ in range(3))
    try:
        # a step so small that t stands still before the ray's end: every ray
        # runs to the loop cap, through empty space
        de.upload(np.tile(np.array([0.1, 0.5, 0.5, 1.0], np.float32), (h, w, 1)))
        dx.upload(np.tile(np.array([0.9, 0.5, 0.5, 1.0], np.float32), (h, w, 1)))
        p = H.default_params(1e-9, kernel=H.KERNEL_CELL, batch=2)   # two lanes per ray: 32 rays per wavefront
        p.loop_cap = cap
        print(f"[case] counters: {w * h} rays of {cap} samples", flush=True)
        st = ctx.render_device(v, t, de, dx, w, h, p, do, stats=True)
        assert st["rays"] == w * h
        assert st["samples"] == w * h * cap
        assert st["lane_slots"] >= st["samples"]
    finally:
        for b in (de, dx, do):
            b.free()
        v.close()
        t.close()
