"""The fused training update and the fused forward pass give the bits of the
layer-by-layer products: batches of one and of several 256-sample chunks, the
largest batch of the fused form and one beyond it, and row counts that leave
half a wave."""
import numpy as np
import pytest

from tiralib_amd import _lib, api
from tiralib_amd._lib import DeviceArray

pytestmark = pytest.mark.gpu


def _rows(src, first, count, width, dtype):
    d = DeviceArray((count, width), dtype)
    _lib.call("tira_hip_memcpy", d.ptr, src.ptr + first * width * d.dtype.itemsize, d.nbytes)
    return d


@pytest.mark.parametrize("batch", [256, 768, 4096, 16384, 16640])
def test_training_equals_single_steps(hip, batch):
    """tira_plate_mlp_train (fused updates) against the same schedule of
    tira_plate_mlp_step calls (one launch per layer and direction)."""
    steps, epochs, lr, lr_final = 3, 2, 1e-2, 1e-4
    a = api.PlateMLP(2.0, 0.5, 2, 16, seed=31)
    a.train(nsamples=steps * batch + 100, epochs=epochs, batch=batch, lr=lr, lr_final=lr_final, seed=77)
    b = api.PlateMLP(2.0, 0.5, 2, 16, seed=31)
    b.set_affine(*a.affine())
    X, T, _ = b.samples(steps * batch, seed=77)
    total = steps * epochs
    warm = min(200, total // 10 + 1)
    lr, fl = np.float32(lr), float(np.float32(lr_final)) / float(np.float32(lr))
    for it in range(total):
        f = (it + 1) / warm if it < warm else fl + (1 - fl) * 0.5 * (1 + np.cos(np.pi * (it - warm) / (total - warm)))
        s = it % steps
        x, t = _rows(X, s * batch, batch, 32, np.uint16), _rows(T, s * batch, batch, 8, np.float32)
        b.step(x, t, np.float32(float(lr) * f))
        x.free()
        t.free()
    np.testing.assert_array_equal(a.params(), b.params())


@pytest.mark.parametrize("rows", [32, 64, 96, 4128])
def test_forward_rows_do_not_depend_on_the_batch(hip, rows):
    net = api.PlateMLP(1.5, 0.0, 1, 16, seed=5)
    X, _, _ = net.samples(8192, seed=6)
    full = net.forward(X).to_host()
    x = _rows(X, 0, rows, 32, np.uint16)
    np.testing.assert_array_equal(net.forward(x).to_host(), full[:rows])


@pytest.mark.parametrize("nsamples", [256, 16640, 65536, 131072])
def test_output_standardisation(hip, nsamples):
    """Means and deviations of the first 65536 training targets against FP64 sums in
    sample order: sums of n terms in another order differ by at most n ulp of FP64,
    7e-12 relative to the sum of magnitudes, so the FP32 results by one rounding."""
    net = api.PlateMLP(1.5, 0.5, 1, 16, seed=8)
    net.train(nsamples=nsamples, epochs=1, batch=256, seed=21)
    _, T, _ = net.samples(nsamples, seed=21)
    t = T.to_host().reshape(nsamples, 8)[:65536, :6].astype(np.float64)
    mu = t.mean(0)
    sd = np.maximum(np.sqrt(np.maximum((t * t).mean(0) - mu * mu, 0)), 1e-3 * (np.abs(mu) + 1e-3))
    got = net.affine()
    np.testing.assert_allclose(got[0], mu, rtol=2.0 ** -23, atol=1e-11 * np.abs(t).max())
    np.testing.assert_allclose(got[1], sd, rtol=2.0 ** -22)
