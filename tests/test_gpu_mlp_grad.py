"""Gradient and Adam step of the stepping network at row counts around the
16-row tile and the workgroup limit, against the oracle and against the step
computed from the gradient."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SEG = {"W1": (0, 1024), "b1": (1024, 1088), "W2": (1088, 5184), "b2": (5184, 5248), "W3": (5248, 5376),
       "b3": (5376, 5378)}


@pytest.mark.parametrize("rows", [1, 15, 16, 17, 100, 4095, 4097, 9000])
def test_gradient_and_step(ctx, oracle, rows):
    from voreen_amd import hipdvr as H
    print(f"[case] mlp gradient and step, {rows} rows", flush=True)
    r = np.random.default_rng(rows)
    p = (r.standard_normal(5378) * 0.2).astype(np.float32)
    x = r.random((rows, 16)).astype(np.float32)
    t = np.stack([r.integers(0, 2, rows), r.random(rows) * 3, r.random(rows)], axis=1).astype(np.float32)
    m = H.Mlp(ctx, seed=8)
    dx, dt = ctx.alloc(x.nbytes), ctx.alloc(t.nbytes)
    try:
        m.set_params(p)
        g, loss = m.gradient(x, t)
        g2, loss2 = m.gradient(x, t)
        assert np.array_equal(g, g2) and loss == loss2   # sums in a fixed order
        lref, gref = oracle.mlp_loss_grad(p.astype(np.float64), x, t, quantize=True)
        # as the repository's gradient test: dZ and the activations are BF16
        assert abs(loss - lref) < 0.01 * abs(lref)
        for name, (a, b) in SEG.items():
            gg, rr = g[a:b].astype(np.float64), gref[a:b]
            rel = np.linalg.norm(gg - rr) / max(np.linalg.norm(rr), 1e-12)
            assert rel < 0.05, f"{name}: {rel:.3g}"
        dx.upload(x)
        dt.upload(t)
        lr = 1e-3
        assert m.train_step_device(dx, dt, rows, lr, want_loss=True) == loss
        # first Adam step: m/c1 = g, v/c2 = g^2 up to a few roundings (1 - 0.999f
        # and c2 agree to 2^-24 / 1e-3)
        g64 = g.astype(np.float64)
        want = p - lr * g64 / (np.abs(g64) + 1e-8)
        got = m.params()
        assert np.abs(got - want).max() <= lr * 1e-3 + np.abs(p).max() * 2.0 ** -23
        # and the packed weights are the new ones
        y = m.forward(x[:100])
        ref = oracle.mlp_forward(got, x[:100], quantize=True)
        assert np.abs(y - ref).max() < 0.03 * max(1.0, np.abs(ref).max())
        g3, _ = m.gradient(x, t)
        _, gref = oracle.mlp_loss_grad(got.astype(np.float64), x, t, quantize=True)
        assert np.linalg.norm(g3 - gref) < 0.05 * np.linalg.norm(gref)
    finally:
        m.close()
        dx.free()
        dt.free()
