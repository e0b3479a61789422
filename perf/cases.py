"""The workloads whose speed this framework is judged by.

Each case is one thing a user's program has the framework do, called through
its public entry points over the sizes, data and options of real use:

    vote2     one 2D stick (+ plate) vote of a host image, the drop-in module call
    search2   a parameter search: many 2D votes of one bound field
    vote3     one 3D vote of a device volume (stick + plate or analytical), with
              or without the eigenvalues of the voted field
    mlp_vote  one 3D vote with the learned plate
    mlp_train training a learned plate for new scales
    eig3      eigenvalues of many tensor arrays in one call
    batch     Gaussian smoothing + eigenvalues of many uneven volumes
    pipeline  intensity volume -> structure tensor -> Gaussian -> vote -> saliency
    skeleton  voted volume -> saliency -> Otsu threshold -> Lee-thinned skeleton

`listed()` holds the named cases, `draw(rng)` one more of the same ranges,
`prepare` / `run` / `work` / `tolerance` / `exact` take a case (a dict of
plain values). Lengths are in voxels; s2 is the fastest axis of a volume.
"""
from __future__ import annotations

import ctypes as C
import math
import random

import numpy as np
import torch

from tiralib_amd import _lib, api, tensorvote_tk

PACKED6, MAT9 = _lib.LAYOUT_PACKED6, _lib.LAYOUT_MAT9


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest call: a 256^2 image of curves, stick votes only, arrays on the host
        # (the module call that a script makes once per image)
        dict(name="vote2_image", kind="vote2", s0=256, s1=256, sigma1=3.0, sigma2=0.0, power=1, w=19, plate=False,
             samples=20),
        # part of one generation of a search over sigma1 in [1, 30], sigma2 in [0, 20] and
        # power in [1, 30] on a bound field: large windows, high powers
        dict(name="search2_generation", kind="search2", s0=256, s1=256, members=12, population=42, samples=20),
        # a small, uneven region of interest: launches and latency
        dict(name="vote3_small", kind="vote3", s0=40, s1=48, s2=56, sigma1=1.5, sigma2=0.0, power=1, w=9,
             atv=False, mat9_in=True, mat9_out=True, eig=False),
        # the ordinary volume: tubes and sheets, sigma 2, vote and eigenvalues in one call
        dict(name="vote3_eig_128", kind="vote3", s0=128, s1=128, s2=128, sigma1=2.0, sigma2=0.0, power=1, w=13,
             atv=False, mat9_in=True, mat9_out=False, eig=True),
        # a narrower vote (power 2) with a second scale on an odd-sized volume
        dict(name="vote3_power2_odd", kind="vote3", s0=91, s1=117, s2=101, sigma1=2.0, sigma2=1.0, power=2, w=13,
             atv=False, mat9_in=False, mat9_out=False, eig=False),
        # analytical voting, ragged
        dict(name="atv3_ragged", kind="vote3", s0=100, s1=150, s2=122, sigma1=2.5, sigma2=0.0, power=1, w=15,
             atv=True, mat9_in=True, mat9_out=False, eig=False),
        # the learned plate at full size: 256^3 curved sheets, sigma 4
        dict(name="mlp_vote_256", kind="mlp_vote", s0=256, s1=256, s2=256, sigma1=4.0, w=25),
        # a new network for sigma 2, from initial weights to the error table
        dict(name="mlp_train_sigma2", kind="mlp_train", sigma1=2.0, sigma2=0.0, power=1, log2_samples=18, epochs=4,
             batch=4096),
        # eigenvalues of uneven volumes, one call
        dict(name="eig3_volumes", kind="eig3", volumes=24, lo=32, hi=256, population=1003, refine=True),
        # smoothing + eigenvalues of 48 uneven volumes, edges 32 .. 256
        dict(name="batch_48_volumes", kind="batch", volumes=48, lo=32, hi=256, population=1003, taps=11, smooth=1.5),
        # the largest: a whole vascular volume from intensity to saliency
        dict(name="pipeline_512", kind="pipeline", s0=384, s1=512, s2=512, smooth=2.0, sigma1=4.0, w=25, tubes=60),
        # the consumer of a vote: threshold and skeleton of a vascular volume
        dict(name="skeleton_256", kind="skeleton", s0=192, s1=256, s2=256, tubes=40),
    ]


def _between(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _eighths(rng, lo, hi):
    """A scale from lo to hi in steps of 1/8 (exact in 32 bits)."""
    return rng.randint(int(lo * 8), int(hi * 8)) / 8.0


def draw(rng):
    kind = rng.choice(["vote2", "search2", "vote3", "vote3", "vote3", "mlp_vote", "mlp_train", "eig3", "batch",
                       "pipeline", "skeleton"])
    if kind == "vote2":
        s1 = _eighths(rng, 1, 5)
        return dict(kind=kind, s0=_between(rng, 48, 640), s1=_between(rng, 48, 640), sigma1=s1,
                    sigma2=rng.choice([0.0, 0.0, s1 / 2]), power=rng.choice([1, 1, 2, 5]), w=2 * int(3 * s1) + 1,
                    plate=rng.random() < 0.5, samples=20)
    if kind == "search2":
        return dict(kind=kind, s0=_between(rng, 96, 320), s1=_between(rng, 96, 320), members=rng.randint(3, 8),
                    population=rng.randint(1, 10 ** 6), samples=rng.choice([10, 20]))
    if kind == "vote3":
        s1 = _eighths(rng, 1, 3.5)
        atv = rng.random() < 0.25
        power = 1 if atv else rng.choice([1, 1, 1, 2, 3])
        top = 160 if power == 1 else 112
        return dict(kind=kind, s0=_between(rng, 20, top), s1=_between(rng, 20, top), s2=_between(rng, 20, top),
                    sigma1=s1, sigma2=0.0 if atv else rng.choice([0.0, 0.0, s1 / 2]), power=power,
                    w=2 * int(3 * s1) + 1, atv=atv, mat9_in=rng.random() < 0.5, mat9_out=rng.random() < 0.5,
                    eig=not atv and rng.random() < 0.3)
    if kind == "mlp_vote":
        s1 = _eighths(rng, 1.5, 3)
        return dict(kind=kind, s0=_between(rng, 32, 160), s1=_between(rng, 32, 160), s2=_between(rng, 32, 160),
                    sigma1=s1, w=2 * int(3 * s1) + 1)
    if kind == "mlp_train":
        return dict(kind=kind, sigma1=_eighths(rng, 1, 2.5), sigma2=rng.choice([0.0, 0.0, 0.5]),
                    power=rng.choice([1, 1, 2]), log2_samples=rng.randint(15, 18), epochs=rng.randint(1, 4),
                    batch=256 * rng.choice([1, 3, 8, 16, 16, 32]))
    if kind in ("eig3", "batch"):
        hi = rng.choice([96, 160, 256])
        c = dict(kind=kind, volumes=rng.randint(2, 24), lo=17, hi=hi, population=rng.randint(1, 10 ** 6))
        if kind == "eig3":
            return dict(c, refine=rng.random() < 0.5)
        taps = rng.choice([5, 7, 9, 11])
        return dict(c, taps=taps, smooth=(taps - 1) / 6.0)
    if kind == "pipeline":
        s1 = _eighths(rng, 1.5, 4)
        return dict(kind=kind, s0=_between(rng, 40, 256), s1=_between(rng, 40, 256), s2=_between(rng, 40, 256),
                    smooth=rng.choice([1.0, 1.5, 2.0]), sigma1=s1, w=2 * int(3 * s1) + 1, tubes=24)
    return dict(kind=kind, s0=_between(rng, 48, 192), s1=_between(rng, 48, 256), s2=_between(rng, 48, 256), tubes=24)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _axis_grids(shape, dtype=torch.float32):
    """Coordinates (x, y, z) = (s2, s1, s0) axes of a volume, broadcastable."""
    z, y, x = (torch.arange(n, device="cuda", dtype=dtype) for n in shape)
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _unit3(r):
    v = [r.gauss(0, 1) for _ in range(3)]
    n = math.sqrt(sum(c * c for c in v)) or 1.0
    return [c / n for c in v]


def _outer6(x, y, z):
    return torch.stack([x * x, x * y, x * z, y * y, y * z, z * z], dim=-1)


def _tubes_and_sheets(shape, seed):
    """Packed-6 field: thin planes (I - n n^T), straight and ring-shaped tubes of
    radius 2 (t t^T), isotropic noise on 1% of the voxels, zero elsewhere."""
    r = random.Random(seed)
    x, y, z = _axis_grids(shape)
    ext = (shape[2], shape[1], shape[0])
    t = torch.zeros(*shape, 6, device="cuda")
    ident = torch.tensor([1.0, 0, 0, 1, 0, 1], device="cuda")
    for _ in range(4):
        n = _unit3(r)
        p = [r.uniform(0.2, 0.8) * e for e in ext]
        m = ((x - p[0]) * n[0] + (y - p[1]) * n[1] + (z - p[2]) * n[2]).abs() <= 0.5
        t[m] = ident - _outer6(*[torch.tensor(c, device="cuda") for c in n])
    for _ in range(8):
        d = _unit3(r)
        p = [r.uniform(0.1, 0.9) * e for e in ext]
        a, b, c = x - p[0], y - p[1], z - p[2]
        along = a * d[0] + b * d[1] + c * d[2]
        t[a * a + b * b + c * c - along * along <= 4.0] = _outer6(*[torch.tensor(v, device="cuda") for v in d])
    for _ in range(8):
        n = _unit3(r)
        p = [r.uniform(0.2, 0.8) * e for e in ext]
        rad = r.uniform(0.1, 0.35) * min(ext)
        a, b, c = torch.broadcast_tensors(x - p[0], y - p[1], z - p[2])
        h = a * n[0] + b * n[1] + c * n[2]
        u, v, w = a - h * n[0], b - h * n[1], c - h * n[2]
        rho = (u * u + v * v + w * w).sqrt()
        m = ((rho - rad) ** 2 + h * h <= 4.0) & (rho > 0.5)
        u, v, w, rho = u[m], v[m], w[m], rho[m]
        t[m] = _outer6((n[1] * w - n[2] * v) / rho, (n[2] * u - n[0] * w) / rho, (n[0] * v - n[1] * u) / rho)
    g = _gen(seed)
    m = torch.rand(shape, device="cuda", generator=g) < 0.01
    mag = 0.5 * torch.rand(shape, device="cuda", generator=g)
    t[m] = mag[m][:, None] * ident
    return t


def _curved_sheets(shape, seed):
    """Packed-6 field of curved sheets (I - n n^T) and 2% plate noise m (I - q q^T)."""
    r = random.Random(seed)
    x, y, z = _axis_grids(shape)
    ext = (shape[2], shape[1], shape[0])
    ident = torch.tensor([1.0, 0, 0, 1, 0, 1], device="cuda")
    t = torch.zeros(*shape, 6, device="cuda")
    for _ in range(12):
        n = _unit3(r)
        u = _unit3(r)
        k = sum(a * b for a, b in zip(u, n))
        u = [a - k * b for a, b in zip(u, n)]
        k = math.sqrt(sum(a * a for a in u))
        u = [a / k for a in u]
        v = [n[1] * u[2] - n[2] * u[1], n[2] * u[0] - n[0] * u[2], n[0] * u[1] - n[1] * u[0]]
        p = [r.uniform(0.2, 0.8) * e for e in ext]
        ka, kb = r.uniform(-0.01, 0.01), r.uniform(-0.01, 0.01)
        a, b, c = torch.broadcast_tensors(x - p[0], y - p[1], z - p[2])
        qu = a * u[0] + b * u[1] + c * u[2]
        qv = a * v[0] + b * v[1] + c * v[2]
        f = a * n[0] + b * n[1] + c * n[2] - ka * qu * qu - kb * qv * qv
        gu, gv = -2 * ka * qu, -2 * kb * qv
        gn = (gu * gu + gv * gv + 1).sqrt()
        m = (f.abs() <= 0.5 * gn) & (qu * qu + qv * qv <= (0.35 * min(shape)) ** 2)
        gu, gv, gn = gu[m], gv[m], gn[m]
        t[m] = ident - _outer6(*[(u[i] * gu + v[i] * gv + n[i]) / gn for i in range(3)])
    g = _gen(seed)
    m = (torch.rand(shape, device="cuda", generator=g) < 0.02) & (t.abs().sum(-1) == 0)
    k = int(m.sum())
    q = torch.nn.functional.normalize(torch.randn(k, 3, device="cuda", generator=g), dim=1)
    mag = 0.5 * torch.rand(k, device="cuda", generator=g)
    t[m] = mag[:, None] * (ident - _outer6(q[:, 0], q[:, 1], q[:, 2]))
    return t


def _segments(shape, count, seed, r_lo, r_hi):
    """Tapered vessel segments: start, direction, length, radii."""
    r = random.Random(seed)
    ext = (shape[2], shape[1], shape[0])
    out = []
    for _ in range(count):
        a = r.uniform(r_lo, r_hi)
        out.append(([r.uniform(0.05, 0.95) * e for e in ext], _unit3(r), r.uniform(0.15, 0.5) * max(ext), a,
                    a * r.uniform(0.7, 1.0)))
    return out


def _vessels(shape, tubes, seed):
    """Intensity 1 inside tapered tubes of radius 2 .. 8, 0 outside, noise of deviation 0.1."""
    x, y, z = _axis_grids(shape)
    v = torch.zeros(shape, device="cuda")
    for p, d, length, ra, rb in _segments(shape, tubes, seed, 2.0, 8.0):
        a, b, c = x - p[0], y - p[1], z - p[2]
        t = (a * d[0] + b * d[1] + c * d[2]).clamp_(0.0, length)
        dist = (a - t * d[0]) ** 2 + (b - t * d[1]) ** 2 + (c - t * d[2]) ** 2
        v[dist <= (ra + t * ((rb - ra) / length)) ** 2] = 1.0
    return v.add_(torch.randn(shape, device="cuda", generator=_gen(seed)), alpha=0.1)


def _voted_vessels(shape, tubes, seed):
    """Packed-6 field as a vote of a vascular volume leaves it: sticks that fall
    off away from the centrelines on a weak ball background with noise."""
    x, y, z = _axis_grids(shape)
    f = torch.zeros(*shape, 6, device="cuda")
    for p, d, length, ra, rb in _segments(shape, tubes, seed, 2.0, 6.0):
        a, b, c = x - p[0], y - p[1], z - p[2]
        t = (a * d[0] + b * d[1] + c * d[2]).clamp_(0.0, length)
        dist = (a - t * d[0]) ** 2 + (b - t * d[1]) ** 2 + (c - t * d[2]) ** 2
        wgt = torch.exp(-dist / (ra + t * ((rb - ra) / length)) ** 2)
        f += wgt[..., None] * _outer6(*[torch.tensor(v, device="cuda") for v in d])
    g = _gen(seed)
    ball = 0.02 * torch.rand(shape, device="cuda", generator=g)
    for k in (0, 3, 5):
        f[..., k] += ball
    return f.add_(torch.randn(f.shape, device="cuda", generator=g), alpha=0.003)


def _mat9(t6):
    return t6[..., [0, 1, 2, 1, 3, 4, 2, 4, 5]].contiguous()


def _image(s0, s1, seed):
    """(H, W, 4) host field: t t^T along cubic Bezier curves, noise sticks on 2% of the pixels."""
    r = np.random.default_rng(seed)
    f = np.zeros((s0, s1, 4), np.float32)

    def put(iy, ix, q, m):
        f[iy, ix] = (m * np.stack([q[0] * q[0], q[0] * q[1], q[0] * q[1], q[1] * q[1]])).T

    for _ in range(8):
        p = r.uniform(0, [s1, s0], size=(4, 2))
        t = np.linspace(0.0, 1.0, 8 * (s0 + s1))[:, None]
        c = (1 - t) ** 3 * p[0] + 3 * (1 - t) ** 2 * t * p[1] + 3 * (1 - t) * t * t * p[2] + t ** 3 * p[3]
        d = (1 - t) ** 2 * (p[1] - p[0]) + 2 * (1 - t) * t * (p[2] - p[1]) + t * t * (p[3] - p[2])
        d /= np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-12)
        i = np.rint(c).astype(int)
        ok = (i[:, 0] >= 0) & (i[:, 0] < s1) & (i[:, 1] >= 0) & (i[:, 1] < s0)
        put(i[ok, 1], i[ok, 0], d[ok].T, 1.0)
    k = r.choice(s0 * s1, size=(s0 * s1) // 50, replace=False)
    th = r.uniform(0, np.pi, k.size)
    put(k // s1, k % s1, np.stack([np.cos(th), np.sin(th)]), r.uniform(0, 0.5, k.size))
    return f


def _members(case):
    """Parameters (sigma1, sigma2, power) of a search generation."""
    r = random.Random(case["population"])
    return [(_eighths(r, 1, 30), _eighths(r, 0, 20), r.randint(1, 30)) for _ in range(case["members"])]


def _shapes(case):
    """Edges of the uneven volumes of a batch: a multiple of 16 or an odd length."""
    r = random.Random(case["population"])
    lo, hi = case["lo"], case["hi"]
    odd = lo % 16 != 0
    return [tuple(r.randint(lo, hi) if odd and r.random() < 0.5 else 16 * r.randint(-(-lo // 16), hi // 16)
                  for _ in range(3)) for _ in range(case["volumes"])]


def _tensors(n, seed):
    """n packed-6 tensors: eigenvalues log-uniform in [1e-3, 1e2], a tenth of them with
    a close pair (relative gap 1e-7 .. 1e-4), random orientation."""
    g = _gen(seed)
    out = torch.empty(n, 6, device="cuda")
    step = 1 << 24
    for a in range(0, n, step):
        k = min(step, n - a)
        lam = torch.exp(torch.rand(k, 3, device="cuda", generator=g, dtype=torch.float64) * math.log(1e5) - math.log(1e3))
        close = torch.rand(k, device="cuda", generator=g) < 0.1
        gap = 10.0 ** (torch.rand(k, device="cuda", generator=g, dtype=torch.float64) * 3 - 7)
        lam[:, 1] = torch.where(close, lam[:, 0] * (1 + gap), lam[:, 1])
        q = torch.randn(k, 4, device="cuda", generator=g, dtype=torch.float64)
        w, x, y, z = (q / q.norm(dim=1, keepdim=True)).unbind(1)
        rows = [(1 - 2 * (y * y + z * z), 2 * (x * y - w * z), 2 * (x * z + w * y)),
                (2 * (x * y + w * z), 1 - 2 * (x * x + z * z), 2 * (y * z - w * x)),
                (2 * (x * z - w * y), 2 * (y * z + w * x), 1 - 2 * (x * x + y * y))]
        for j, (p, s) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
            out[a:a + k, j] = sum(rows[p][m] * rows[s][m] * lam[:, m] for m in range(3)).float()
    return out


def _vol(case):
    return case["s0"], case["s1"], case["s2"]


# ------------------------------------------------------------------ prepare
class _Buf:
    """A torch tensor as the framework's Python calls take a device buffer."""

    def __init__(self, t):
        self.t, self.ptr, self.shape = t, t.data_ptr(), tuple(t.shape)


class _Batch:
    """The handle of a batched launch with the buffers it was made for."""

    def __init__(self, case, seed):
        shapes = _shapes(case)
        n = [a * b * c for a, b, c in shapes]
        at = np.concatenate([[0], np.cumsum(n)])
        self.src = _tensors(int(at[-1]), seed)
        self.out = torch.empty_like(self.src)
        self.ev = torch.empty(int(at[-1]), 3, device="cuda")
        torch.cuda.synchronize()
        P = C.c_void_p * len(n)
        self.args = [P(*[t.data_ptr() + 4 * t.shape[1] * int(a) for a in at[:-1]]) for t in (self.src, self.out, self.ev)]
        edges = np.ascontiguousarray(shapes, np.uint32)
        taps = api.gaussian_taps(case["taps"], case["smooth"])
        h = C.c_void_p()
        _lib.call("tira_batch_gauss_eig3_create", C.byref(h), len(n), *[C.cast(a, C.c_void_p) for a in self.args],
                  edges.ctypes.data, taps.ctypes.data, taps.size, 1)
        self.handle = h.value

    def __del__(self):
        if getattr(self, "handle", None):
            _lib.call("tira_batch_gauss_eig3_destroy", self.handle)
            self.handle = None


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "vote2":
        s["field"] = _image(case["s0"], case["s1"], seed)
    elif kind == "search2":
        s["session"] = tensorvote_tk.Session(_image(case["s0"], case["s1"], seed))
        s["members"] = _members(case)
    elif kind == "vote3":
        t = _tubes_and_sheets(_vol(case), seed)
        s["field"] = _Buf(_mat9(t) if case["mat9_in"] else t)
        s["out"] = _Buf(torch.empty(*_vol(case), 9 if case["mat9_out"] else 6, device="cuda"))
        s["ev"] = torch.empty(*_vol(case), 3, device="cuda") if case["eig"] else None
    elif kind == "mlp_vote":
        s["field"] = _Buf(_curved_sheets(_vol(case), seed))
        s["out"] = _Buf(torch.empty(*_vol(case), 6, device="cuda"))
        s["net"] = api.PlateMLP(case["sigma1"], 0.0, 1, 64, seed=1004)
        s["net"].train(nsamples=1 << 18, epochs=4, batch=4096, seed=1004)
    elif kind == "mlp_train":
        s["seed"] = int(seed)
    elif kind == "eig3":
        sizes = [a * b * c for a, b, c in _shapes(case)]
        s["src"] = _tensors(sum(sizes), seed)
        s["ev"] = torch.empty(sum(sizes), 3, device="cuda")
        s["in"] = [_Buf(t) for t in s["src"].split(sizes)]
        s["out"] = [_Buf(t) for t in s["ev"].split(sizes)]
        s["counts"] = sizes
    elif kind == "batch":
        s["batch"] = _Batch(case, seed)
    elif kind == "pipeline":
        s["volume"] = _Buf(_vessels(_vol(case), case["tubes"], seed))
        s["saliency"] = _Buf(torch.empty(*_vol(case), 3, device="cuda"))
    elif kind == "skeleton":
        s["voted"] = _voted_vessels(_vol(case), case["tubes"], seed)
        s["saliency"] = torch.empty(*_vol(case), 3, device="cuda")
        s["threshold"] = torch.empty(1, device="cuda")
        s["skeleton"] = torch.empty(_vol(case), dtype=torch.uint8, device="cuda")
    else:
        raise ValueError(f"unknown kind {kind!r}")
    return s


# ------------------------------------------------------------------ run
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "vote2":
        return tensorvote_tk.tensorvote_tk(s["field"], case["sigma1"], case["sigma2"], case["power"], case["w"], True,
                                           case["plate"], case["samples"])
    if kind == "search2":
        return [s["session"].tensorvote_tk(a, b, p, samples=case["samples"]) for a, b, p in s["members"]]
    if kind == "vote3":
        shape, lin, lout = _vol(case), MAT9 if case["mat9_in"] else PACKED6, MAT9 if case["mat9_out"] else PACKED6
        if case["atv"]:
            api.tensorvote3_atv_async(s["field"], s["out"], shape, case["sigma1"], case["w"], in_layout=lin,
                                      out_layout=lout)
        elif case["eig"]:
            _lib.call("tira_tensorvote3_eig_async", s["field"].ptr, lin, s["out"].ptr, lout, *shape, case["sigma1"],
                      case["sigma2"], case["w"], case["power"], 1, 1, 20, _lib.PLATE_AUTO, s["ev"].data_ptr(),
                      _lib.EIG_REFINE_FP64 | _lib.EIG_SCALE_INVARIANT, None)
            return s["out"].t, s["ev"]
        else:
            api.tensorvote3_async(s["field"], s["out"], shape, case["sigma1"], case["sigma2"], case["w"],
                                  case["power"], in_layout=lin, out_layout=lout)
        return s["out"].t
    if kind == "mlp_vote":
        s["net"].vote(s["field"], s["out"], _vol(case), case["w"], tol=0.5, in_layout=PACKED6)
        return s["out"].t
    if kind == "mlp_train":
        net = api.PlateMLP(case["sigma1"], case["sigma2"], case["power"], 64, seed=s["seed"])
        net.train(nsamples=1 << case["log2_samples"], epochs=case["epochs"], batch=case["batch"], seed=s["seed"] + 1)
        out = {"params": net.params(), "table_errors": net.table_errors(), "table": net.vote_table()[0]}
        net.close()
        return out
    if kind == "eig3":
        flags = _lib.EIG_SCALE_INVARIANT | (_lib.EIG_REFINE_FP64 if case["refine"] else 0)
        api.eig3_batch(s["in"], counts=s["counts"], evals=s["out"], flags=flags)
        return s["ev"]
    if kind == "batch":
        b = s["batch"]
        _lib.call("tira_batch_gauss_eig3_run", b.handle)
        return b.out, b.ev
    if kind == "pipeline":
        api.pipeline3(s["volume"], smooth_sigma=case["smooth"], vote_sigma=case["sigma1"], w=case["w"],
                      saliency=s["saliency"])
        return s["saliency"].t
    it = C.c_uint()
    _lib.call("tira_skeleton3", s["voted"].data_ptr(), PACKED6, *_vol(case), s["saliency"].data_ptr(),
              s["threshold"].data_ptr(), s["skeleton"].data_ptr(), C.byref(it))
    return s["saliency"], s["threshold"], s["skeleton"], int(it.value)


# ------------------------------------------------------------------ work, tolerance
def _pairs(shape, w):
    r, p = w // 2, 1
    for n in shape:
        p *= sum(min(n - 1, i + r) - max(0, i - r) + 1 for i in range(n))
    return p


def work(case):
    """What a pass cannot do without: its inputs read and its results written once,
    and the arithmetic of the formulation that needs least of it."""
    kind = case["kind"]
    if kind in ("vote2", "search2"):
        n = case["s0"] * case["s1"]
        if kind == "vote2":
            return {"bytes": 32 * n, "flops": _pairs((case["s0"], case["s1"]), case["w"]) * (32 if case["plate"] else 26)}
        w = [2 * int(3 * max(a, b)) + 1 for a, b, _ in _members(case)]
        return {"bytes": 16 * n * (1 + case["members"]), "flops": 32 * sum(_pairs((case["s0"], case["s1"]), k) for k in w)}
    if kind == "mlp_train":
        # forward, backward and weight gradients of 53k FLOP a sample, in 64 B + 32 B a sample
        k = (1 << case["log2_samples"]) // case["batch"] * case["batch"] * case["epochs"]
        return {"bytes": 96 * k, "flops": 53000 * k}
    if kind in ("eig3", "batch"):
        n = sum(a * b * c for a, b, c in _shapes(case))
        return {"bytes": n * (36 if kind == "eig3" else 60), "flops": n * (150 + (36 * case["taps"] if kind == "batch" else 0))}
    n = case["s0"] * case["s1"] * case["s2"]
    # a vote of degree g = 2 p + 2 as a correlation of its (g + 1)(g + 2) / 2 features, through
    # real FFTs of the padded volume
    g = 2 * case.get("power", 1) + 2
    nf = (g + 1) * (g + 2) // 2
    pad = 1
    for k in ("s0", "s1", "s2"):
        pad *= case.get(k, 1) + case.get("w", 0) // 2
    fft = pad * (2.5 * math.log2(pad) * (nf + 6) + 6 * nf)
    if kind == "vote3":
        return {"bytes": n * ((36 if case["mat9_in"] else 24) + (36 if case["mat9_out"] else 24) + (12 if case["eig"] else 0)),
                "flops": fft}
    if kind == "mlp_vote":
        return {"bytes": 48 * n, "flops": 63 * _pairs(_vol(case), case["w"])}
    if kind == "pipeline":
        k = 2 * (int(math.ceil(6 * case["smooth"])) // 2) + 1
        return {"bytes": 16 * n, "flops": fft + n * (36 * k + 170)}
    return {"bytes": 37 * n, "flops": 200 * n}


def tolerance(case):
    kind = case["kind"]
    if kind == "mlp_train":
        # 16-bit activations through hundreds of updates: another order of the sums moves the weights
        return {"rel": 0.02, "max": 0.9}
    if kind == "mlp_vote":
        return {"rel": 5e-6, "max": 1e-3}
    if kind == "skeleton":
        return {"rel": 2e-6, "max": 1e-4, "differ": 1e-5}
    if kind in ("eig3", "batch"):
        return {"rel": 2e-6, "max": 1e-4}
    return {"rel": 5e-6, "max": 1e-4}


# ------------------------------------------------------------------ exact: 64 bits, plain torch
def _jacobi3(t6):
    """Eigenvalues (ascending, list of 3) and eigenvectors (list of 3 lists of 3) of
    packed-6 tensors by cyclic Jacobi rotations in 64 bits."""
    t = t6.double()
    a = {(0, 0): t[..., 0].clone(), (0, 1): t[..., 1].clone(), (0, 2): t[..., 2].clone(), (1, 1): t[..., 3].clone(),
         (1, 2): t[..., 4].clone(), (2, 2): t[..., 5].clone()}
    one, zero = torch.ones_like(a[0, 0]), torch.zeros_like(a[0, 0])
    v = [[one.clone() if i == j else zero.clone() for j in range(3)] for i in range(3)]  # v[column][row]
    for _ in range(6):
        for p, q, k in ((0, 1, 2), (0, 2, 1), (1, 2, 0)):
            apq = a[p, q]
            live = apq != 0
            tau = (a[q, q] - a[p, p]) / (2 * torch.where(live, apq, one))
            tan = torch.where(tau >= 0, 1.0, -1.0) / (tau.abs() + torch.sqrt(1 + tau * tau))
            tan = torch.where(live, tan, zero)
            c = torch.rsqrt(1 + tan * tan)
            s = tan * c
            kp, kq = tuple(sorted((k, p))), tuple(sorted((k, q)))
            a[p, p], a[q, q] = a[p, p] - tan * apq, a[q, q] + tan * apq
            a[p, q] = zero
            a[kp], a[kq] = c * a[kp] - s * a[kq], s * a[kp] + c * a[kq]
            for r in range(3):
                v[p][r], v[q][r] = c * v[p][r] - s * v[q][r], s * v[p][r] + c * v[q][r]
    lam = [a[0, 0], a[1, 1], a[2, 2]]
    for i, j in ((0, 1), (1, 2), (0, 1)):
        swap = lam[i] > lam[j]
        lam[i], lam[j] = torch.where(swap, lam[j], lam[i]), torch.where(swap, lam[i], lam[j])
        for r in range(3):
            v[i][r], v[j][r] = torch.where(swap, v[j][r], v[i][r]), torch.where(swap, v[i][r], v[j][r])
    return lam, v


def _fast_length(n):
    while True:
        k = n
        for f in (2, 3, 5):
            while k % f == 0:
                k //= f
        if k == 1:
            return n
        n += 1


def _atten(l2, sigma):
    return (l2 <= 1e-12).double() if sigma == 0 else torch.exp(-l2 / (sigma * sigma))


def _correlate(features, kernels, shape, reach):
    """sum_f sum_d K_{c,f}(d) F_f(x + d): features yields (F_f, [K_c,f over the window])."""
    L = [_fast_length(n + r) for n, r in zip(shape, reach)]
    acc = None
    at = [torch.arange(-r, r + 1, device="cuda") % k for r, k in zip(reach, L)]
    where = torch.meshgrid(*at, indexing="ij")
    dims = tuple(range(len(shape)))
    for f, ks in zip(features, kernels):
        F = torch.fft.rfftn(f, s=L, dim=dims)
        if acc is None:
            acc = [torch.zeros_like(F) for _ in ks]
        for c, k in enumerate(ks):
            w = torch.zeros(L, dtype=torch.float64, device="cuda")
            w[where] = k
            acc[c] += torch.fft.rfftn(w, dim=dims).conj() * F
        del F
    cut = tuple(slice(0, n) for n in shape)
    return [torch.fft.irfftn(x, s=L, dim=dims)[cut] for x in acc]


def _stick3(d, c1, c2, power, q):
    """Stick votes of unit q (..., 3) over offsets d (..., 3): six components."""
    t = (q * d).sum(-1)
    eta = c1 * (1 - t * t) ** power + c2 * t ** (2 * power)
    r = q - 2 * t[..., None] * d
    return eta[..., None] * _outer6(r[..., 0], r[..., 1], r[..., 2])


def _atv3(d, c, T, inv):
    """c R H R with H = T - inv (v^T T v T + 2 T v v^T T), R = I - 2 d d^T, of symmetric T (..., 3, 3)."""
    tv = (T @ d[..., None])[..., 0]
    H = T - inv * ((d * tv).sum(-1)[..., None, None] * T + 2 * tv[..., :, None] * tv[..., None, :])
    R = torch.eye(3, device="cuda", dtype=torch.float64) - 2 * d[..., :, None] * d[..., None, :]
    V = R @ H @ R * c[..., None, None]
    return torch.stack([V[..., 0, 0], V[..., 0, 1], V[..., 0, 2], V[..., 1, 1], V[..., 1, 2], V[..., 2, 2]], -1)


def _vote3(t6, shape, sigma1, sigma2, power, w, atv):
    """The 3D vote of a packed-6 field: votes are polynomials of even degree g in an
    eigenvector on the unit sphere, fitted exactly per offset, then correlated."""
    lam, vec = _jacobi3(t6)
    h = w // 2
    r = torch.arange(-h, h + 1, device="cuda", dtype=torch.float64)
    dw, dv, du = torch.meshgrid(r, r, r, indexing="ij")
    l2 = du * du + dv * dv + dw * dw
    il = torch.where(l2 > 0, torch.rsqrt(torch.where(l2 > 0, l2, torch.ones_like(l2))), torch.zeros_like(l2))
    d = torch.stack([du * il, dv * il, dw * il], -1).reshape(-1, 1, 3)
    c1, c2 = _atten(l2, sigma1).reshape(-1, 1), _atten(l2, sigma2).reshape(-1, 1)
    g = 4 if atv else 2 * power + 2
    expo = [(a, b, g - a - b) for a in range(g + 1) for b in range(g + 1 - a)]
    rng = np.random.default_rng(0)
    q = rng.normal(size=(4 * len(expo), 3))
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    mono = np.stack([q[:, 0] ** a * q[:, 1] ** b * q[:, 2] ** c for a, b, c in expo], 1)
    fit = torch.from_numpy(np.linalg.pinv(mono)).cuda()  # (nf, M)
    q = torch.from_numpy(q).cuda()[None]
    W = 2 * h + 1

    def window(votes):  # (offsets, M, 6) -> (6, nf, W, W, W)
        return torch.einsum("omc,fm->cfo", votes, fit).reshape(6, len(expo), W, W, W)

    def features(weight, e):
        for a, b, c in expo:
            yield weight * e[0] ** a * e[1] ** b * e[2] ** c

    ident = torch.eye(3, device="cuda", dtype=torch.float64)
    if atv:
        qq = q[..., :, None] * q[..., None, :]
        parts = [(lam[2] - lam[1], vec[2], window(_atv3(d, c1, qq, 1 / 3))),
                 (lam[1] - lam[0], vec[0], window(_atv3(d, c1, ident - qq, 1 / 4))),
                 (lam[0], None, _atv3(d[:, 0], c1[:, 0], ident, 1 / 5).T.reshape(6, 1, W, W, W))]
    else:
        f = math.factorial
        sn = 1.0 / (math.pi ** 1.5 / 2 * (sigma1 ** 3 * 2.0 ** (2 * power + 1) * f(power) ** 2 / f(2 * power + 1)
                                          + sigma2 ** 3 * 2.0 / (2 * power + 1)))
        ref = torch.where(q[..., 2:].abs() < 0.9, ident[2], ident[0])
        u = torch.nn.functional.normalize(torch.linalg.cross(ref, q), dim=-1)
        v = torch.linalg.cross(q, u)
        m = 2 * power + 4  # equispaced samples integrate the polynomial over the circle exactly
        plate = sum(_stick3(d, c1, c2, power, math.cos(math.pi * i / m) * u + math.sin(math.pi * i / m) * v)
                    for i in range(m)) * (math.pi / m)
        parts = [(torch.copysign(lam[2].abs() - lam[1].abs(), lam[2]), vec[2], sn * window(_stick3(d, c1, c2, power, q))),
                 (torch.copysign(lam[1].abs() - lam[0].abs(), lam[1]), vec[0], window(plate) / math.pi)]

    def all_features():
        for wgt, e, _ in parts:
            if e is None:
                yield wgt
            else:
                yield from features(wgt, e)

    kernels = [k[:, i] for _, _, k in parts for i in range(k.shape[1])]
    return torch.stack(_correlate(all_features(), kernels, shape, (h, h, h)), -1)


def _vote2(field, sigma1, sigma2, power, w, plate, samples):
    """The 2D vote of an (H, W, 4) field: even harmonics of the stick's angle, correlated."""
    t = torch.from_numpy(field).cuda().double()
    a, b, c = t[..., 0], t[..., 1], t[..., 3]
    mean, rad = 0.5 * (a + c), torch.hypot(0.5 * (a - c), b)
    l0, l1 = mean - rad, mean + rad
    theta = 0.5 * torch.atan2(2 * b, a - c)
    h = w // 2
    r = torch.arange(-h, h + 1, device="cuda", dtype=torch.float64)
    dv, du = torch.meshgrid(r, r, indexing="ij")
    l2 = du * du + dv * dv
    il = torch.where(l2 > 0, torch.rsqrt(torch.where(l2 > 0, l2, torch.ones_like(l2))), torch.zeros_like(l2))
    dx, dy = du * il, dv * il
    c1, c2 = _atten(l2, sigma1), _atten(l2, sigma2)
    norm = 1.0
    for k in range(1, power + 1):
        norm *= 2.0 * k / (2 * k - 1)
    norm /= math.pi * (sigma1 * sigma1 + sigma2 * sigma2)

    def stick(th):
        qx, qy = math.cos(th), math.sin(th)
        tt = qx * dx + qy * dy
        eta = norm * (c1 * (1 - tt * tt) ** power + c2 * tt ** (2 * power))
        x, y = qx - 2 * tt * dx, qy - 2 * tt * dy
        return [eta * x * x, eta * x * y, eta * y * y]

    m = 2 * power + 6
    at = [math.pi * j / m for j in range(m)]
    votes = [stick(th) for th in at]
    weight = torch.copysign(l1.abs() - l0.abs(), l1)
    feats, kernels = [], []
    for k in range(power + 2):
        for fn, tf in ((math.cos, torch.cos), (math.sin, torch.sin)):
            if k == 0 and fn is math.sin:
                continue
            feats.append(weight * tf(2 * k * theta))
            kernels.append([(1.0 if k == 0 else 2.0) / m * sum(v[i] * fn(2 * k * th) for v, th in zip(votes, at))
                            for i in range(3)])
    if plate:
        v = [stick(math.pi / samples * i) for i in range(samples)]
        feats.append(l0)
        kernels.append([sum(x[i] for x in v) * (math.pi / samples) for i in range(3)])
    x = _correlate(feats, kernels, l0.shape, (h, h))
    return torch.stack([x[0], x[1], x[1], x[2]], -1).cpu().numpy()


def _smooth(t, taps, sigma):
    """Zero-padded separable Gaussian of (s0, s1, s2, C) in 64 bits."""
    h = taps // 2
    k = [math.exp(-0.5 * (i / sigma) ** 2) for i in range(-h, h + 1)]
    k = [v / sum(k) for v in k]
    t = t.double()
    for axis in range(3):
        n = t.shape[axis]
        o = torch.zeros_like(t)
        for i in range(-h, h + 1):
            m = n - abs(i)
            if m > 0:
                o.narrow(axis, max(0, -i), m).add_(t.narrow(axis, max(0, i), m), alpha=k[i + h])
        t = o
    return t


def _structure(v):
    g = []
    for axis in (2, 1, 0):
        n = v.shape[axis]
        d = torch.empty_like(v)
        d.narrow(axis, 1, n - 2).copy_((v.narrow(axis, 2, n - 2) - v.narrow(axis, 0, n - 2)) / 2)
        d.narrow(axis, 0, 1).copy_(v.narrow(axis, 1, 1) - v.narrow(axis, 0, 1))
        d.narrow(axis, n - 1, 1).copy_(v.narrow(axis, n - 1, 1) - v.narrow(axis, n - 2, 1))
        g.append(d)
    return _outer6(*g)


def exact(case, seed):
    kind = case["kind"]
    if kind == "vote2":
        return _vote2(_image(case["s0"], case["s1"], seed), case["sigma1"], case["sigma2"], case["power"], case["w"],
                      case["plate"], case["samples"])
    if kind == "search2":
        f = _image(case["s0"], case["s1"], seed)
        return [_vote2(f, a, b, p, 2 * int(3 * max(a, b)) + 1, True, case["samples"]) for a, b, p in _members(case)]
    if kind == "vote3":
        o = _vote3(_tubes_and_sheets(_vol(case), seed), _vol(case), case["sigma1"], case["sigma2"], case["power"],
                   case["w"], case["atv"])
        v = _mat9(o) if case["mat9_out"] else o
        return (v, torch.stack(_jacobi3(o)[0], -1)) if case["eig"] else v
    if kind == "eig3":
        t = _tensors(sum(a * b * c for a, b, c in _shapes(case)), seed)
        return torch.cat([torch.stack(_jacobi3(x)[0], -1) for x in t.split(1 << 24)])
    if kind == "batch":
        sizes = _shapes(case)
        t = _tensors(sum(a * b * c for a, b, c in sizes), seed)
        out, ev = [], []
        for x, s in zip(t.split([a * b * c for a, b, c in sizes]), sizes):
            out.append(_smooth(x.reshape(*s, 6), case["taps"], case["smooth"]).reshape(-1, 6))
            ev.append(torch.stack(_jacobi3(x)[0], -1))
        return torch.cat(out), torch.cat(ev)
    if kind == "pipeline":
        t = _structure(_vessels(_vol(case), case["tubes"], seed).double())
        k = int(math.ceil(6 * case["smooth"]))
        t = _smooth(t, k + (k % 2 == 0), case["smooth"])
        o = _vote3(t, _vol(case), case["sigma1"], 0.0, 1, case["w"], False)
        del t
        l = _jacobi3(o)[0]
        return torch.stack([l[2] - l[1], l[1] - l[0], l[0]], -1)
    if kind == "skeleton":
        lam = _jacobi3(_voted_vessels(_vol(case), case["tubes"], seed))[0]
        m = torch.stack([x.abs() for x in lam], -1).sort(-1).values
        return torch.stack([m[..., 2] - m[..., 1], m[..., 1] - m[..., 0], m[..., 0]], -1), None, None, None
    return None  # a trained network has no value of its own in 64 bits
