"""Device-built pre-integration tables at sizes around the kernel's runs and
diagonal groups, read back entry by entry through two-sample rays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 4, 5, 31, 33, 64, 257, 513])
@pytest.mark.parametrize("kind", ["random", "sparse"])
def test_device_table_equals_the_host_table(ctx, n, kind):
    from voreen_amd import hipdvr as H, workloads as W
    print(f"[case] preint table n={n} {kind}", flush=True)
    keys = (W.random_keys(n, 7) if kind == "random" else
            [(0.0, (9, 200, 30, 0)), (0.4, (9, 200, 30, 0)), (0.5, (250, 10, 90, 255)), (0.6, (20, 250, 90, 0)),
             (1.0, (255, 255, 0, 0))])
    r = np.random.default_rng(n)
    vol = ctx.volume(r.integers(0, 65536, (32, 32, 32)).astype(np.uint16))
    tf = ctx.transfunc(np.full((2, 4), 255, np.uint8))
    w, h, step = 256, 256, 0.4
    # rays of two samples `step` apart, each at a random voxel
    en = np.ones((h, w, 4), np.float32)
    ex = np.ones((h, w, 4), np.float32)
    en[..., :3] = r.random((h, w, 3)) * 0.3
    d = r.random((h, w, 3)) + 0.2
    ex[..., :3] = en[..., :3] + 1.5 * step * d / np.linalg.norm(d, axis=2, keepdims=True)
    out = {}
    try:
        for name in ("device", "host"):
            if name == "device":
                tf.preint_device(keys, n, 0.003)
            else:
                tf.set_preint(H.preint_build(keys, n, 0.003))
            p = H.default_params(step, classification=H.CLASS_PREINT, filter_=H.FILTER_NEAREST)
            out[name], st = ctx.render(vol, tf, en, ex, p)
            assert w * h <= st["samples"] <= 2 * w * h
    finally:
        tf.close()
        vol.close()
    diff = np.abs(out["device"] - out["host"]).max(axis=2)
    # alpha and the premultiplied colour gather at most one rounding of the
    # power (two ulps at 1) per step; the un-premultiplied colour divides by
    # alpha >= 0.001, where steps are few and small, and is weighted by it again
    tol = 8 * n * 2.0 ** -24
    assert np.mean(diff > tol) < 1e-3, f"max {diff.max():.3g}"
    # an entry whose alpha meets 0.95 within a rounding stops a step earlier or
    # later: one sample behind 0.95
    assert diff.max() <= 0.06


def test_largest_table_of_one_colour(ctx):
    """n = 4096, one colour of alpha 0.2: every entry is that colour with
    alpha 1 - 0.8 ** (200 step)."""
    from voreen_amd import hipdvr as H
    print("[case] preint table n=4096 one colour", flush=True)
    n, step, w, h = 4096, 0.4, 128, 128
    r = np.random.default_rng(1)
    vol = ctx.volume(r.integers(0, 65536, (32, 32, 32)).astype(np.uint16))
    tf = ctx.transfunc(np.full((2, 4), 255, np.uint8))
    en = np.ones((h, w, 4), np.float32)
    ex = np.ones((h, w, 4), np.float32)
    en[..., :3] = r.random((h, w, 3)) * 0.3
    ex[..., :3] = en[..., :3] + 0.9   # 1.56 long: four samples
    try:
        tf.preint_device([(0.0, (255, 102, 51, 51)), (1.0, (255, 102, 51, 51))], n, 0.003)
        img, st = ctx.render(vol, tf, en, ex, H.default_params(step, classification=H.CLASS_PREINT,
                                                               filter_=H.FILTER_NEAREST))
    finally:
        tf.close()
        vol.close()
    assert st["samples"] == 4 * w * h
    a = 1.0 - 0.8 ** 0.6   # of one entry; 4096 steps of at most two roundings at 1 each
    A = 1.0 - (1.0 - a) ** 4
    want = np.array([A, A * 0.4, A * 0.2, A])
    assert np.abs(img - want).max() <= 4 * 4096 * 2 * 2.0 ** -24
