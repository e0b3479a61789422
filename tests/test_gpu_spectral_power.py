"""The spectral vote of powers 2 to 4 (28, 45, 66 features) against the window
gather and, at one receiver set, the FP64 oracle: every combination of stick,
plate, input and layout, sizes that are odd, ragged and larger than one row
block, and the voters that have to be voted by window instead."""
import numpy as np
import pytest

from tiralib_amd import _lib, api, synth

pytestmark = pytest.mark.gpu
SLOTS = [0, 1, 2, 4, 5, 8]


def _field(shape, seed):
    f = synth.tubes_sheets_volume(shape, n_straight=3, n_helix=2, n_sheets=2, seed=seed).reshape(shape + (9,))
    rng = np.random.default_rng(seed)
    a = rng.normal(size=shape + (3, 3)) * (rng.random(shape) < 0.05)[..., None, None]  # signed, all three eigenvalues
    return np.ascontiguousarray(f + (a + a.swapaxes(-1, -2)).reshape(shape + (9,)), np.float32)


def _run(f, shape, mode, sigma, sigma2, w, power, stick=True, plate=True, samples=20, out_layout=_lib.LAYOUT_MAT9):
    d, o = _lib.DeviceArray.from_host(f), _lib.DeviceArray(shape + (9 if out_layout == _lib.LAYOUT_MAT9 else 6,))
    try:
        _lib.call("tira_hip_profile_begin")
        api.tensorvote3_async(d, o, shape, sigma, sigma2, w, power, stick=stick, plate=plate, samples=samples,
                              plate_mode=mode, out_layout=out_layout)
        _lib.call("tira_hip_synchronize")
        _lib.call("tira_hip_profile_end")
        return o.to_host(), _lib.profile_get("spec_mul")[1]
    finally:
        d.free()
        o.free()


def _rel(a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("power", [2, 3, 4])
@pytest.mark.parametrize("shape,w,stick,plate,samples,layout", [
    ((32, 32, 32), 11, True, True, 20, _lib.LAYOUT_MAT9),
    ((33, 41, 37), 11, True, False, 0, _lib.LAYOUT_PACKED6),
    ((19, 50, 71), 13, False, True, 6, _lib.LAYOUT_MAT9),
    ((3, 90, 129), 13, True, True, 0, _lib.LAYOUT_PACKED6),
])
def test_spectral_power_equals_gather(hip, power, shape, w, stick, plate, samples, layout):
    f = _field(shape, seed=power)
    got, n = _run(f, shape, _lib.PLATE_AUTO, 2.0, 1.0, w, power, stick, plate, samples, layout)
    ref, m = _run(f, shape, _lib.PLATE_CLOSED, 2.0, 1.0, w, power, stick, plate, samples, layout)
    assert (n, m) == (1, 0)
    # either is within 1e-6 of 64 bits at these windows (5e-7 .. 1e-6 measured)
    assert _rel(got, ref) <= 2e-6


@pytest.mark.parametrize("power", [2, 3, 4])
def test_spectral_power_vs_oracle(hip, oracle, power):
    shape, w = (34, 32, 35), 11
    f = _field(shape, seed=11)
    rng = np.random.default_rng(1)
    recv = np.sort(rng.choice(int(np.prod(shape)), 200, replace=False))
    ref = oracle.tensorvote3_f64(f, 1.75, 0.5, power, w, samples=20, recv=recv, nthreads=8)[:, SLOTS]
    got, n = _run(f, shape, _lib.PLATE_AUTO, 1.75, 0.5, w, power)
    assert n == 1
    assert _rel(got.reshape(-1, 9)[recv][:, SLOTS], ref) <= 4e-6  # sampled: four times the whole field's 1e-6


@pytest.mark.parametrize("power,w,spectral", [(2, 7, 0), (2, 9, 1), (3, 9, 1), (4, 9, 0), (4, 11, 1), (5, 13, 0)])
def test_spectral_power_rule(hip, power, w, spectral):
    shape = (32, 32, 32)
    f = _field(shape, seed=2)
    for mode in (_lib.PLATE_AUTO, _lib.VOTE_SPECTRAL):
        assert _run(f, shape, mode, 1.5, 0.0, w, power)[1] == spectral
    assert _run(f, shape, _lib.PLATE_AUTO, 1.5, 0.0, w, power, samples=power + 1)[1] == 0  # not the exact integral


@pytest.mark.parametrize("bad", [np.nan, np.inf, 3e37])
def test_wild_voter_is_voted_by_window(hip, bad):
    """A voter that the transforms would spread or overflow leaves the gather's result."""
    shape = (32, 36, 40)
    f = _field(shape, seed=4)
    f[12, 20, 17] = 0
    f[12, 20, 17, 0] = bad
    got, n = _run(f, shape, _lib.PLATE_AUTO, 1.5, 0.0, 9, 2)
    ref, _ = _run(f, shape, _lib.PLATE_CLOSED, 1.5, 0.0, 9, 2)
    assert n == 1
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
    inside = np.zeros(shape, bool)
    inside[8:17, 16:25, 13:22] = True
    assert np.isfinite(got[~inside]).all()
    assert np.abs(got[~inside] - ref[~inside]).max() <= 1e-5 * np.abs(ref[~inside]).max()
    a, b = got[inside], ref[inside]
    ok = np.isfinite(b)
    assert ok.sum() == 0 or np.abs(a[ok] - b[ok]).max() <= 1e-5 * np.abs(b[ok]).max()


def test_stick_of_other_length_is_voted_by_window(hip):
    """Eigenvectors handed in need not be of unit length: the vote takes them as they are."""
    shape = (32, 33, 34)
    n = int(np.prod(shape))
    rng = np.random.default_rng(5)
    e = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0].astype(np.float32)
    lam = np.sort(rng.random((n, 3)), axis=1).astype(np.float32)
    e2, e0 = np.ascontiguousarray(e[:, :, 0]), np.ascontiguousarray(e[:, :, 1])
    out = {}
    for name, scale in (("unit", 1.0), ("long", 1.5)):
        for power in (2,):
            out[name] = api.tensorvote3_tk(lam, e2 * np.float32(scale), e0, shape, 1.5, 0.0, power, 9, True, False, 20)
    # (1 - t^2)^p of a longer vector is no multiple of the unit one's: check against one receiver in 64 bits
    at, h = (16, 17, 18), 4
    for name, scale in (("unit", 1.0), ("long", 1.5)):
        V = np.zeros((3, 3))
        q3 = (e2.reshape(shape + (3,)) * scale).astype(np.float64)
        l3 = lam.reshape(shape + (3,)).astype(np.float64)
        sn = 1 / (np.pi ** 1.5 / 2 * 1.5 ** 3 * 2 ** 5 * 4 / 120)
        for dw in range(-h, h + 1):
            for dv in range(-h, h + 1):
                for du in range(-h, h + 1):
                    l2 = du * du + dv * dv + dw * dw
                    d = np.array([du, dv, dw]) / np.sqrt(l2) if l2 else np.zeros(3)
                    i = (at[0] + dw, at[1] + dv, at[2] + du)
                    q, s = q3[i], l3[i][2] - l3[i][1]
                    t = q @ d
                    eta = np.exp(-l2 / 1.5 ** 2) * (1 - t * t) ** 2 + (t ** 4 if l2 == 0 else 0)
                    r = q - 2 * t * d
                    V += sn * s * eta * np.outer(r, r)
        g = out[name].reshape(shape + (3, 3))[at]
        assert np.abs(g - V).max() <= 1e-5 * np.abs(V).max(), name


@pytest.mark.parametrize("power", [2, 3, 4])
@pytest.mark.parametrize("normal", [(0, 0, 1), (0, 1, 0), (1, 0, 0), (0, .6, .8), (.6, .8, 0), (.8, 0, .6), (.48, .6, .64)])
@pytest.mark.parametrize("scale", [1e38, 3e36])
def test_wild_plate_is_voted_by_window(hip, power, normal, scale):
    """A finite plate whose features overflow (all of them to NaN where the normal has
    a zero component) leaves the rest of the volume as the window gather has it."""
    shape, w, at = (32, 34, 36), 11, (15, 16, 17)
    f = _field(shape, seed=5)
    n = np.array(normal, np.float64)
    f[at] = (scale * (np.eye(3) - np.outer(n, n))).astype(np.float32).ravel()
    got, _ = _run(f, shape, _lib.PLATE_AUTO, 2.0, 0.0, w, power)
    ref, _ = _run(f, shape, _lib.PLATE_CLOSED, 2.0, 0.0, w, power)
    inside = np.zeros(shape, bool)
    inside[tuple(slice(c - w // 2, c + w // 2 + 1) for c in at)] = True
    assert np.isfinite(ref[~inside]).all()
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
    assert np.abs(got[~inside].astype(np.float64) - ref[~inside]).max() <= 1e-5 * np.abs(ref[~inside]).max()


@pytest.mark.parametrize("power", [2, 3, 4])
@pytest.mark.parametrize("bad", [np.inf, np.nan, 3e38])
def test_wild_eigenvalue_is_voted_by_window(hip, power, bad):
    """The same through eigenpair input, plates only and sticks only."""
    shape, w, at = (32, 34, 36), 11, (15, 16, 17)
    n = int(np.prod(shape))
    rng = np.random.default_rng(power)
    e = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0]
    e[np.ravel_multi_index(at, shape)] = np.eye(3)  # zero components
    e2, e0 = (np.ascontiguousarray(e[:, :, k], np.float32) for k in (0, 1))
    lam = np.sort(rng.random((n, 3)), axis=1).astype(np.float32)
    lam[np.ravel_multi_index(at, shape)] = 0
    inside = np.zeros(shape, bool)
    inside[tuple(slice(c - w // 2, c + w // 2 + 1) for c in at)] = True
    for stick, plate in ((False, True), (True, False)):
        clean = api.tensorvote3_tk(lam, e2, e0, shape, 1.5, 0.0, power, w, stick, plate, 20).reshape(shape + (9,))
        l = lam.copy()
        l[np.ravel_multi_index(at, shape), 1 if plate else 2] = bad
        got = api.tensorvote3_tk(l, e2, e0, shape, 1.5, 0.0, power, w, stick, plate, 20).reshape(shape + (9,))
        assert np.isfinite(got[~inside]).all()
        assert np.abs(got[~inside].astype(np.float64) - clean[~inside]).max() <= 1e-5 * np.abs(clean[~inside]).max()


@pytest.mark.parametrize("power", [2, 3, 4])
@pytest.mark.parametrize("length", [1e20, 3e38, 1e-7])
def test_plate_of_a_normal_beyond_range(hip, power, length):
    """A caller's normal whose squared length leaves FP32 becomes the zero vector, which
    has no circle of directions to vote along: its plate stays within its window."""
    shape, w, at = (32, 34, 36), 11, (15, 16, 17)
    n, i = int(np.prod(shape)), np.ravel_multi_index(at, shape)
    rng = np.random.default_rng(power)
    e0 = np.ascontiguousarray(np.linalg.qr(rng.normal(size=(n, 3, 3)))[0][:, :, 1], np.float32)
    lam = np.sort(rng.random((n, 3)), axis=1).astype(np.float32)
    lam[i] = 0
    inside = np.zeros(shape, bool)
    inside[tuple(slice(c - w // 2, c + w // 2 + 1) for c in at)] = True
    clean = api.tensorvote3_tk(lam, None, e0, shape, 1.5, 0.0, power, w, False, True, 20).reshape(shape + (9,))
    lam[i], e0[i] = (0.0, 1.0, 1.0), (0.0, length, 0.0)
    got = api.tensorvote3_tk(lam, None, e0, shape, 1.5, 0.0, power, w, False, True, 20).reshape(shape + (9,))
    assert np.isfinite(got[~inside]).all()
    assert np.abs(got[~inside].astype(np.float64) - clean[~inside]).max() <= 1e-5 * np.abs(clean[~inside]).max()


@pytest.mark.parametrize("wild", [False, True])
@pytest.mark.parametrize("power", [2, 4])
def test_input_may_lie_in_the_output(hip, power, wild):
    """Eigenpairs in the memory of the output, and a field voted in place: as with an
    output of its own, also where a voter has the field voted by window."""
    shape, w = (32, 33, 35), 11
    n = int(np.prod(shape))
    rng = np.random.default_rng(7)
    e = np.linalg.qr(rng.normal(size=(n, 3, 3)))[0].astype(np.float32)
    lam = np.sort(rng.random((n, 3)), axis=1).astype(np.float32)
    f = _field(shape, seed=9).reshape(n, 9)
    if wild:
        lam[n // 2] = np.inf
        f[n // 2] = np.inf
    parts = np.concatenate([lam.ravel(), e[:, :, 0].ravel(), e[:, :, 1].ravel()])
    one, own, two = _lib.DeviceArray.from_host(parts), _lib.DeviceArray((n, 9)), _lib.DeviceArray.from_host(f)
    try:
        src = [one.ptr + 12 * n * k for k in range(3)]
        for out in (own.ptr, one.ptr):
            _lib.call("tira_tensorvote3_tk", out, *src, *shape, 1.5, 0.0, power, w, 1, 1, 20)
        np.testing.assert_array_equal(one.to_host().reshape(n, 9), own.to_host())
        assert np.isfinite(own.to_host()).any()
        for out in (own, two):
            api.tensorvote3_async(two, out, shape, 1.5, 0.0, w, power)
        _lib.call("tira_hip_synchronize")
        np.testing.assert_array_equal(two.to_host(), own.to_host())
    finally:
        for d in (one, own, two):
            d.free()


@pytest.mark.parametrize("power,w", [(2, 9), (3, 9), (4, 11)])
@pytest.mark.parametrize("bright", [1.0, 1e3, 1e6])
def test_faint_votes_beside_a_bright_voter(hip, oracle, power, w, bright):
    """The vote of faint voters keeps its digits where a bright voter stands elsewhere
    in the field: receivers outside its window, against the window gather (whose
    rounding knows nothing of it) and, one by one, against FP64. Transforms in FP32
    lose 1e-10 of the bright voter: 1e-4 of these votes at 1e6."""
    shape, at = (36, 40, 44), (4, 5, 6)
    f = _field(shape, seed=8)
    f[tuple(slice(0, c + w) for c in at)] = 0
    f[at] = bright * np.diag([1.0, 0.25, 0.0]).astype(np.float32).ravel()
    got, n = _run(f, shape, _lib.PLATE_AUTO, 1.5, 0.0, w, power)
    ref, _ = _run(f, shape, _lib.PLATE_CLOSED, 1.5, 0.0, w, power)
    assert n == 1
    far = np.ones(shape, bool)
    far[tuple(slice(0, c + w // 2 + 1) for c in at)] = False
    assert _rel(got[far], ref[far]) <= 2e-6
    # receiver by receiver, down to a thousandth of the largest of these votes
    size = np.linalg.norm(ref, axis=-1)
    strong = np.flatnonzero(far & (size > 1e-3 * size[far].max()))
    recv = np.sort(np.random.default_rng(3).choice(strong, 300, replace=False))
    exact = oracle.tensorvote3_f64(f, 1.5, 0.0, power, w, samples=20, recv=recv, nthreads=8)
    err = np.linalg.norm(got.reshape(-1, 9)[recv].astype(np.float64) - exact, axis=1) / np.linalg.norm(exact, axis=1)
    # a voter's FP32 direction enters a vote 2 p + 2 times, 6e-8 each, and votes of opposite
    # sign cancel to a sixth of their magnitudes at most where they are this large
    assert err.max() <= (2 * power + 2) * 6e-8 * 6


@pytest.mark.parametrize("power", [2, 3, 4])
def test_spectral_power_is_closer_to_64_bits_than_the_gather(hip, oracle, power):
    shape, w = (32, 35, 33), 11
    f = _field(shape, seed=13)
    rng = np.random.default_rng(2)
    recv = np.sort(rng.choice(int(np.prod(shape)), 300, replace=False))
    ref = oracle.tensorvote3_f64(f, 2.0, 1.0, power, w, samples=20, recv=recv, nthreads=8)[:, SLOTS]
    err = [_rel(_run(f, shape, mode, 2.0, 1.0, w, power)[0].reshape(-1, 9)[recv][:, SLOTS], ref)
           for mode in (_lib.PLATE_AUTO, _lib.PLATE_CLOSED)]
    # voters and result in FP32, all between in FP64: a few roundings of 6e-8, averaged over the voters
    assert err[0] <= min(err[1], 1.2e-7)


@pytest.mark.parametrize("power,w", [(2, 9), (4, 11)])
@pytest.mark.parametrize("bright", [1e10, 1e12, 1e30, 3e37])
def test_range_beyond_fp64_is_voted_by_window(hip, power, w, bright):
    """A voter so bright that even FP64 transforms would cost the others digits:
    the whole field is the window gather's, bit for bit."""
    shape, at = (33, 34, 35), (4, 5, 6)
    f = _field(shape, seed=8)
    f[at] = bright * np.diag([1.0, 0.25, 0.0]).astype(np.float32).ravel()
    got, _ = _run(f, shape, _lib.PLATE_AUTO, 1.5, 0.0, w, power)
    ref, _ = _run(f, shape, _lib.PLATE_CLOSED, 1.5, 0.0, w, power)
    np.testing.assert_array_equal(got, ref)
    # scales all as large are no range: the spectral vote, and close to the gather
    g = (_field(shape, seed=8) * np.float32(bright / 1e3)).astype(np.float32)
    got, _ = _run(g, shape, _lib.PLATE_AUTO, 1.5, 0.0, w, power)
    ref, _ = _run(g, shape, _lib.PLATE_CLOSED, 1.5, 0.0, w, power)
    assert not np.array_equal(got, ref) and _rel(got, ref) <= 2e-6
