"""The learned-plate vote over listed voters (plate_sparse.hip) against the
window gather of the same table, on fields whose density, size and window sit
at the edges of the listed form: cubes and tiles cut by the volume's border,
windows wider than an axis, empty fields, dense and mixed tiles.

Handing a network its own vote table back marks the table as the caller's,
which always takes the window gather: the same pairs in another order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plates(shape, density, seed):
    rng = np.random.default_rng(seed)
    n = rng.normal(size=shape + (3,))
    n /= np.linalg.norm(n, axis=-1, keepdims=True)
    x, y, z = n[..., 0], n[..., 1], n[..., 2]
    t = np.stack([1 - x * x, -x * y, -x * z, 1 - y * y, -y * z, 1 - z * z], -1)
    t *= rng.uniform(0.2, 1.0, shape)[..., None]
    on = rng.random(shape) < (density if np.isscalar(density) else density[..., None, None] * np.ones(shape))
    return np.ascontiguousarray(np.where(on[..., None], t, 0), np.float32)


@pytest.fixture(scope="module")
def nets(hip):
    from tiralib_amd import api
    out = {}
    for sigma in (1.5, 2.0):
        a, b = (api.PlateMLP(sigma, 0.0, 1, 64, seed=3) for _ in range(2))
        a.train(nsamples=1 << 14, epochs=2, batch=1024, seed=5)
        b.set_params(a.params())
        b.set_affine(*a.affine())
        b.set_vote_table(a.vote_table()[0])
        out[sigma] = (a, b)
    yield out
    for pair in out.values():
        for n in pair:
            n.close()


def _vote(hip, net, f, w, stick, layout):
    d = hip.DeviceArray.from_host(f)
    o = hip.DeviceArray(f.shape[:3] + (9 if layout == hip.LAYOUT_MAT9 else 6,))
    try:
        net.vote(d, o, f.shape[:3], w, stick=stick, tol=1e30, in_layout=hip.LAYOUT_PACKED6, out_layout=layout)
        hip.call("tira_hip_synchronize")
        return o.to_host()
    finally:
        d.free()
        o.free()


@pytest.mark.parametrize("shape,sigma,w,density", [
    ((1, 1, 1), 1.5, 9, 1.0),
    ((3, 5, 7), 1.5, 9, 0.4),
    ((33, 37, 41), 1.5, 3, 0.05),
    ((33, 37, 65), 2.0, 13, 0.0),
    ((20, 30, 129), 2.0, 13, 0.02),
    ((24, 21, 70), 2.0, 13, 1.0),
    ((61, 18, 67), 1.5, 9, "mixed"),
])
@pytest.mark.parametrize("stick", [False, True])
def test_listed_plates_equal_window_gather(hip, nets, shape, sigma, w, density, stick):
    dens = np.linspace(0, 1, shape[0]) ** 3 if density == "mixed" else density
    f = _plates(shape, dens, seed=sum(shape))
    a, b = nets[sigma]
    layout = hip.LAYOUT_MAT9 if shape[2] % 2 else hip.LAYOUT_PACKED6
    got, ref = _vote(hip, a, f, w, stick, layout), _vote(hip, b, f, w, stick, layout)
    # two orders of up to 13^3 FP32 terms per receiver: each within sqrt(2197) 2^-24 = 2.8e-6
    # of the exact sum in the root mean square
    norm = np.linalg.norm(ref.astype(np.float64))
    assert np.linalg.norm(got.astype(np.float64) - ref) <= 5.6e-6 * norm
    if density == 0.0:
        assert norm == 0 and not got.any()


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_bad_voter_stays_in_its_window(hip, nets, bad):
    """One voter that is not finite spoils its own window and nothing else."""
    f = _plates((40, 36, 44), 0.05, seed=9)
    w, at = 9, (17, 20, 25)
    clean = f.copy()
    clean[at] = 0
    f[at] = bad
    net = nets[1.5][0]
    for stick in (False, True):
        got, ref = _vote(hip, net, f, w, stick, hip.LAYOUT_PACKED6), _vote(hip, net, clean, w, stick, hip.LAYOUT_PACKED6)
        inside = np.zeros(f.shape[:3], bool)
        inside[tuple(slice(c - w // 2, c + w // 2 + 1) for c in at)] = True
        assert np.isfinite(got[~inside]).all()
        # the sticks come from the window gather then, and from the spectral vote without the bad voter
        assert np.abs(got[~inside].astype(np.float64) - ref[~inside]).max() <= 1e-5 * np.abs(ref).max()


@pytest.mark.parametrize("w,density", [(9, 1.0), (9, 0.05), (13, 1.0), (7, 0.05)])
def test_sticks_of_the_learned_vote(hip, nets, w, density):
    """Sticks and plates of fields that the density and the window send to the spectral
    vote with listed or windowed plates (w >= 13, or few plates) or to one window
    gather (bit for bit the caller's table's, which never lists): the same votes."""
    shape = (34, 40, 70)
    f = _plates(shape, density, seed=3)
    rng = np.random.default_rng(4)
    q = rng.normal(size=shape + (3,))
    q /= np.linalg.norm(q, axis=-1, keepdims=True)
    on = (rng.random(shape) < 0.1)[..., None]
    x, y, z = q[..., 0], q[..., 1], q[..., 2]
    f = f + np.where(on, np.stack([x * x, x * y, x * z, y * y, y * z, z * z], -1), 0).astype(np.float32)
    a, b = nets[2.0 if w == 13 else 1.5]
    got, ref = _vote(hip, a, f, w, True, hip.LAYOUT_PACKED6), _vote(hip, b, f, w, True, hip.LAYOUT_PACKED6)
    if w < 9 or (w < 13 and density == 1.0):
        np.testing.assert_array_equal(got, ref)
    # w^3 FP32 terms in either order, as test_listed_plates_equal_window_gather
    assert np.linalg.norm(got.astype(np.float64) - ref) <= 5.6e-6 * np.linalg.norm(ref.astype(np.float64))


@pytest.mark.parametrize("bright", [1e6, 1e12])
def test_faint_sticks_beside_a_bright_one(hip, nets, bright):
    """Receivers outside the window of a bright stick keep the votes of the faint
    ones; a range beyond FP64 sends sticks and plates to the window gather."""
    shape, w, at = (36, 40, 44), 9, (5, 6, 7)
    f = _plates(shape, 0.03, seed=12)
    f[..., 0] += 0.2 * (np.random.default_rng(1).random(shape) < 0.1)  # sticks along x
    f[at] = bright * np.array([1, 0, 0, 0, 0, 0], np.float32)
    a, b = nets[1.5]
    got, ref = _vote(hip, a, f, w, True, hip.LAYOUT_PACKED6), _vote(hip, b, f, w, True, hip.LAYOUT_PACKED6)
    far = np.ones(shape, bool)
    far[tuple(slice(0, c + w // 2 + 1) for c in at)] = False
    d = got[far].astype(np.float64) - ref[far]
    assert np.linalg.norm(d) <= 5.6e-6 * np.linalg.norm(ref[far].astype(np.float64))
    if bright == 1e12:
        np.testing.assert_array_equal(got, ref)
