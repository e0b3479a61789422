"""The spectral votes' offset kernels as the votes use them (fitted, transformed and
multiplied on the device): the field of one voter is its vote at every offset of the
window and nothing outside it, checked against the oracle's FP64 pair votes."""
import itertools

import numpy as np
import pytest

from tiralib_amd import _lib, api

pytestmark = pytest.mark.gpu
SHAPE, AT = (32, 33, 34), (15, 17, 16)
SLOTS = [0, 1, 2, 4, 5, 8]


def _atten(l2, s):
    return np.exp(-l2 / s ** 2) if s > 0 else (0.0 if l2 > 0 else 1.0)


def _vote(tensor, fn):
    f = np.zeros(SHAPE + (9,), np.float32)
    f[AT] = tensor.ravel()
    d, o = _lib.DeviceArray.from_host(f), _lib.DeviceArray(SHAPE + (9,))
    try:
        _lib.call("tira_hip_profile_begin")
        fn(d, o)
        _lib.call("tira_hip_synchronize")
        _lib.call("tira_hip_profile_end")
        assert _lib.profile_get("spec_mul")[1] == 1
        return o.to_host()[..., SLOTS].astype(np.float64)
    finally:
        d.free()
        o.free()


def _compare(got, pair, w, tol):
    r, worst, scale = w // 2, 0.0, 0.0
    out = got.copy()
    for off in itertools.product(range(-r, r + 1), repeat=3):  # dw, dv, du: voter minus receiver
        at = tuple(a - o for a, o in zip(AT, off))
        ref = pair(off[2], off[1], off[0])
        worst, scale = max(worst, np.abs(got[at] - ref).max()), max(scale, np.abs(ref).max())
        out[at] = 0
    assert worst <= tol * scale, worst / scale
    assert np.abs(out).max() <= tol * scale  # nothing outside the window


@pytest.mark.parametrize("power,w,s1,s2", [(1, 7, 1.5, 0.0), (1, 9, 2.0, 1.2), (2, 9, 1.5, 0.0), (2, 9, 2.0, 1.0),
                                           (3, 9, 1.75, 0.5), (4, 11, 2.0, 0.0), (4, 11, 1.5, 2.0)])
@pytest.mark.parametrize("kind", ["stick", "plate"])
def test_vote_of_one_voter(hip, oracle, power, w, s1, s2, kind):
    rng = np.random.default_rng(10 * power + w)
    sn = oracle.sticknorm3(float(np.float32(s1)), float(np.float32(s2)), power)
    for k in range(4):
        q = rng.normal(size=3) if k else np.array([0.0, 0.6, 0.8])
        q /= np.linalg.norm(q)
        t = np.outer(q, q) if kind == "stick" else np.eye(3) - np.outer(q, q)

        def pair(du, dv, dw):
            d = np.array([du, dv, dw], float)
            l2 = float(d @ d)
            d = d / np.sqrt(l2) if l2 else d
            c1, c2 = _atten(l2, s1), _atten(l2, s2)
            if kind == "stick":
                return oracle.stick3_pair_f64(d, c1, c2, power, q) / sn
            return oracle.plate3_sum_f64(d, c1, c2, power, q, 20) / np.pi

        got = _vote(t.astype(np.float32), lambda d, o: api.tensorvote3_async(d, o, SHAPE, s1, s2, w, power))
        # the FP32 tensor's eigenvector is off by 1e-7 and enters 2 p + 2 times; FP32 transforms
        # (power 1) add 1e-6
        _compare(got, pair, w, (2 * power + 2) * 1e-7 + (1e-6 if power == 1 else 0.0))


@pytest.mark.parametrize("w,sigma", [(7, 1.5), (9, 2.5)])
def test_atv_of_one_voter(hip, oracle, w, sigma):
    rng = np.random.default_rng(w)
    for _ in range(3):
        e = np.linalg.qr(rng.normal(size=(3, 3)))[0]
        lam = np.array([0.3, 1.1, 2.4])
        t = ((e * lam) @ e.T).astype(np.float32)
        got = _vote(t, lambda d, o: api.tensorvote3_atv_async(d, o, SHAPE, sigma, w))

        def pair(du, dv, dw):
            return oracle.atv3_pair(lam, e[:, 1], e[:, 2], (du, dv, dw), sigma, f64=True)[[0, 1, 3, 2, 4, 5]]

        _compare(got, pair, w, 2e-6)
