"""The listed gather of a 2D search session (a field of few voters) against the
module's window gather: tiles cut by the border, windows wider than the field,
even windows, powers around and beyond the squaring's bits, no voter at all,
and the share of voters at which the session changes over."""
import numpy as np
import pytest

import tiralib_amd.tensorvote_tk as tvk
from tiralib_amd import api

pytestmark = pytest.mark.gpu


def _field(shape, share, seed):
    r = np.random.default_rng(seed)
    th, m = r.uniform(0, np.pi, shape), r.uniform(0.2, 1.0, shape)
    l0 = r.uniform(-0.3, 0.3, shape)
    on = np.zeros(shape[0] * shape[1], bool)
    on[r.choice(on.size, int(share * on.size), replace=False)] = True
    m, l0 = m * on.reshape(shape), l0 * on.reshape(shape)
    c, s = np.cos(th), np.sin(th)
    return np.stack([m * c * c + l0, m * c * s, m * c * s, m * s * s + l0], -1).astype(np.float32)


def _close(got, ref, terms):
    # two orders of `terms` FP32 votes: each within sqrt(terms) 2^-24 of the largest sum, in the mean
    bound = 4 * max(np.sqrt(terms), 8) * 2.0 ** -24 * max(np.abs(ref).max(), 1e-30)
    assert np.abs(got - ref).max() <= bound


@pytest.mark.parametrize("shape", [(1, 1), (3, 70), (65, 5), (64, 64), (130, 129), (40, 200)])
@pytest.mark.parametrize("share", [0.0, 0.03, 0.39, 0.6])
def test_listed_session_equals_module(hip, shape, share):
    f = _field(shape, share, sum(shape))
    with tvk.Session(f) as s:
        for k, (s1, s2, p) in enumerate([(1.0, 0.0, 1), (3.0, 1.0, 2), (5.0, 0.0, 7), (4.0, 6.0, 31), (2.0, 2.0, 64)]):
            stick, plate = k % 3 != 1, k % 3 != 2
            got = s.tensorvote_tk(s1, s2, p, stick=stick, plate=plate)
            ref = tvk.tensorvote_tk(f, s1, s2, p, stick=stick, plate=plate)
            _close(got, ref, (2 * int(3 * max(s1, s2)) + 1) ** 2)


def test_listed_session_even_window_and_both_outputs(hip):
    """An even window through the C ABI (it ends at offset w / 2 - 1), host and
    device outputs in turn, and a caller's table in between on the same session."""
    import ctypes as C
    from tiralib_amd._lib import DeviceArray, call
    f = _field((50, 61), 0.1, 7)
    h, out = C.c_void_p(), DeviceArray((50, 61, 4))
    call("tira_vote2_session_create", C.byref(h), f.ctypes.data, 50, 61)
    try:
        for w in (12, 13, 1, 2):
            host = np.empty((50, 61, 4), np.float32)
            call("tira_vote2_session_vote", h, host.ctypes.data, None, 0, 2.5, 1.0, 2, w, 1, 1, 20)
            call("tira_vote2_session_vote", h, out.ptr, None, 0, 2.5, 1.0, 2, w, 1, 1, 20)
            ref = api.tensorvote(f, 2.5, 1.0, 2, w, True, True, 20)
            _close(host, ref, w * w)
            np.testing.assert_array_equal(out.to_host(), host)
            nb = api.build_neighbors2d(w, 2.5, 1.0, 2, 20)
            call("tira_vote2_session_vote", h, host.ctypes.data, nb.ctypes.data, nb.size, 2.5, 1.0, 2, w, 1, 1, 20)
            np.testing.assert_array_equal(host, api.tensorvote_prebuilt(f, nb, 2.5, 1.0, 2, w, True, True, 20))
    finally:
        out.free()
        call("tira_vote2_session_destroy", h)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_listed_session_bad_voter(hip, bad):
    f = _field((48, 80), 0.05, 3)
    f[20, 30] = bad
    with tvk.Session(f) as s:
        got, ref = s.tensorvote_tk(2.0, 1.0, 3), tvk.tensorvote_tk(f, 2.0, 1.0, 3)
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
    ok = np.isfinite(ref)
    _close(got[ok], ref[ok], 13 * 13)


@pytest.mark.parametrize("share", [0.05, 0.7])
def test_session_of_a_device_field_still_being_written(hip, share):
    """A session bound to device memory that work queued on the library's stream
    still has to write (a long kernel ahead of the copy) holds what was written."""
    import ctypes as C
    from tiralib_amd import _lib
    shape = (300, 260)
    f, stale = _field(shape, share, 5), _field(shape, 0.02, 6)
    src, field, busy = _lib.DeviceArray.from_host(f), _lib.DeviceArray.from_host(stale), _lib.DeviceArray((1024,))
    h, st, got = C.c_void_p(), C.c_void_p(), np.empty(shape + (4,), np.float32)
    _lib.call("tira_hip_stream_create", C.byref(st))
    try:
        _lib.call("tira_hip_set_stream", st)
        _lib.call("tira_hip_fma_loop_async", busy.ptr, 1024, 1 << 18)  # tens of milliseconds
        _lib.call("tira_hip_copy_async", field.ptr, src.ptr, f.nbytes)
        _lib.call("tira_vote2_session_create", C.byref(h), field.ptr, *shape)
        for p in (1, 3):
            _lib.call("tira_vote2_session_vote", h, got.ctypes.data, None, 0, 3.0, 1.0, p, 19, 1, 1, 20)
            with tvk.Session(f) as ref:
                np.testing.assert_array_equal(got, ref.tensorvote_tk(3.0, 1.0, p, w=19))
    finally:
        _lib.call("tira_hip_synchronize")
        _lib.call("tira_hip_set_stream", None)
        if h:
            _lib.call("tira_vote2_session_destroy", h)
        _lib.call("tira_hip_stream_destroy", st)
        for d in (src, field, busy):
            d.free()


@pytest.mark.parametrize("share", [0.1, 0.7])
@pytest.mark.parametrize("s1,s2,p", [(14.0, 0.0, 29), (12.0, 2.0, 23), (8.0, 8.0, 30)])
def test_vote_scale_at_high_powers(hip, oracle, share, s1, s2, p):
    """The common scale of a vote at high powers against FP64: the least-squares
    factor between the two fields. What scales all sticks alike is the norm (one
    rounding, 6e-8) and the sums' bias (below one rounding); the float product of p
    ratios that the norm was taken from is 4e-7 off at p = 29."""
    f = _field((48, 56), share, 11)
    w = 2 * int(3 * max(s1, s2)) + 1
    ref = oracle.tensorvote2_f64(f, s1, s2, p, w, True, False, 20, nthreads=8)
    with tvk.Session(f) as s:
        for got in (s.tensorvote_tk(s1, s2, p, w=w, plate=False), tvk.tensorvote_tk(f, s1, s2, p, w=w, plate=False)):
            scale = ((got.astype(np.float64) - ref) * ref).sum() / (ref * ref).sum()
            assert abs(scale) <= (1.3e-7 if s2 == 0.0 else 2.5e-7), scale


@pytest.mark.parametrize("share", [0.19, 0.21, 0.39, 0.41])
def test_share_and_window_pick_the_gather(hip, share):
    """Around the shares and the window at which a session changes over: narrow and
    wide windows in turn on one session, against the module's window gather; where
    the window gather serves them too, to an ulp of a vote with its table."""
    f = _field((90, 110), share, 21)
    with tvk.Session(f) as s:
        for k, (s1, s2, p) in enumerate([(3.0, 0.0, 1), (4.0, 0.0, 2), (3.5, 1.0, 3), (3.0, 0.0, 1), (8.0, 2.0, 4)]):
            w = 2 * int(3 * max(s1, s2)) + 1
            got, ref = s.tensorvote_tk(s1, s2, p), tvk.tensorvote_tk(f, s1, s2, p)
            _close(got, ref, w * w)
            if share > 0.4 or (share > 0.2 and w < 25):
                nb = api.build_neighbors2d(w, s1, s2, p, 20)
                one = s.tensorvote_tk_prebuilt(nb.tobytes(), nb.size, w, s1, s2, p)
                # the device's table may differ from the host's by an ulp in c1, c2
                assert np.abs(got - one).max() <= 1.2e-7 * np.abs(one).max()
