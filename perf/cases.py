"""The workloads whose speed is followed: what a user of shearcuda_amd has it do.

A case is a dict of plain values; ``kind`` names the path it takes:

* ``denoise``   one image, decompose -> hard threshold -> reconstruct
* ``transform`` one image, decomposition and reconstruction as two calls
* ``batch``     many images of one size through one plan
* ``train``     one unrolled shearlet/wavelet shrink iteration, forward and backward
* ``separate``  one iteration of the cartoon / point separation loop
* ``rdwt``      undecimated wavelet transform and its inverse, any size
* ``mad``       noise scalars: median absolute deviation of a stack of planes
* ``volume``    3D denoise of a batch of volumes
* ``bands3d``   3D analysis, its transpose and the band-pass round trip

``prepare`` makes the inputs on the GPU from the seed and the handles a program
keeps; ``run`` is one pass; ``exact`` restates the pass in 64 bits with plain
torch.  The spatial filter tables (Meyer shearing filters, maxflat pyramid, 3D
cone filters) are inputs of the dictionaries, so ``exact`` takes the same tables.

A hard threshold is a jump: a coefficient within rounding of it may fall on
either side, and each such coefficient moves the image by far more than
rounding.  So every hard threshold here is the usual T * sigma * s moved by at
most 5% to the middle of the widest gap between neighbouring magnitudes of its
band, found in 64 bits.  Thresholds of a training pass are placed the same way,
since its gradient has the same jump.
"""
import functools
import math

import numpy as np
import torch

from shearcuda_amd import api, separation, shearlet3d
from shearcuda_amd.filters import dictionary_filters
from shearcuda_amd.filters3d import get_meyer_based_filter
from shearcuda_amd.wavelets import MakeONFilter

DEV = "cuda"
F64 = torch.float64

# dictionaries: directions per scale (log2) and filter sides, coarse to fine
DICTS = {
    "default": ((3, 3, 4, 4), (32, 32, 16, 16)),
    "demo80": ((3, 3, 4, 4), (80, 80, 80, 80)),    # the separation demo's
    "light": ((2, 2, 3, 3), (32, 32, 16, 16)),
    "three": ((3, 3, 4), (32, 32, 16)),
    "narrow": ((2, 3, 3), (24, 16, 16)),
}
WAVELETS = {"haar": ("Haar", 0), "d4": ("Daubechies", 4), "d6": ("Daubechies", 6), "sym4": ("Symmlet", 4)}


# ---- cases -------------------------------------------------------------------------

def listed():
    return [
        # the smallest image: an interactive tool's preview, one eager call
        dict(name="denoise_128", kind="denoise", L=128, dict="default", shift="none", sigma=20.0, coeffs=False,
             tuned=False, graph=False),
        # the headline step: one 512^2 image, tuned plan, replayed graph, image only
        dict(name="denoise_512", kind="denoise", L=512, dict="default", shift="none", sigma=20.0, coeffs=False,
             tuned=True, graph=True),
        # the largest image a dictionary takes, eager, coefficients kept
        dict(name="denoise_1024", kind="denoise", L=1024, dict="default", shift="none", sigma=20.0, coeffs=True,
             tuned=False, graph=False),
        # the two transforms as a program that works on the coefficients calls them
        dict(name="transform_256", kind="transform", L=256, dict="default", shift="center"),
        # a folder of small images, each with its own noise level
        dict(name="batch_256x48", kind="batch", L=256, nimg=48, dict="default", shift="none", coeffs=False,
             tuned=True),
        # large images in a serving loop
        dict(name="batch_1024x8", kind="batch", L=1024, nimg=8, dict="default", shift="none", coeffs=False,
             tuned=True),
        # training learnable thresholds: forward and backward of one unrolled iteration
        dict(name="train_512x8", kind="train", L=512, nimg=8, dict="default", shift="none", levels=3, wavelet="d4",
             tuned=True),
        # the shipped separation demo's iteration, pre-emphasis included
        dict(name="separate_512", kind="separate", L=512, dict="demo80", shift="none", level2=4, tuned=False),
        # wavelet transform of camera frames whose sides are no powers of two
        dict(name="rdwt_4x1000x1496", kind="rdwt", nimg=4, m=1000, n=1496, levels=3, wavelet="sym4"),
        # noise estimation of every band of a 512^2 dictionary
        dict(name="mad_49x512", kind="mad", planes=49, elems=512 * 512, arith="fp64"),
        # the volume workload: 128^3, three levels, 432 bands
        dict(name="volume_128x2", kind="volume", n=128, nvol=2, dirs="8,8,4", mode=1.0),
        # 3D coefficients and their transpose, as an iterative solver calls them
        dict(name="bands3d_64", kind="bands3d", n=64, nvol=1, dirs="4,4,4", mode=1.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["denoise", "denoise", "transform", "batch", "batch", "train", "separate", "rdwt", "mad",
                       "volume", "bands3d"])
    shift = rng.choice(["none", "none", "center"])
    name = rng.choice(["default", "default", "light", "three", "narrow"])
    wavelet = rng.choice(sorted(WAVELETS))
    if kind == "denoise":
        return dict(kind=kind, L=rng.choice([64, 128, 256, 512, 1024]), dict=name, shift=shift,
                    sigma=round(rng.uniform(8.0, 30.0), 2), coeffs=rng.random() < 0.5, tuned=rng.random() < 0.3,
                    graph=rng.random() < 0.4)
    if kind == "transform":
        return dict(kind=kind, L=rng.choice([64, 128, 256, 512, 1024]), dict=name, shift=shift)
    if kind == "batch":
        L = rng.choice([64, 128, 256, 512, 1024])
        return dict(kind=kind, L=L, nimg=_log(rng, 2, min(64, 8 * 1024 ** 2 // L ** 2)), dict=name, shift=shift,
                    coeffs=rng.random() < 0.4, tuned=rng.random() < 0.5)
    if kind == "train":
        L = rng.choice([64, 128, 256, 512])
        return dict(kind=kind, L=L, nimg=_log(rng, 1, min(24, 8 * 512 ** 2 // L ** 2)), dict=name, shift=shift,
                    levels=rng.randint(1, 3), wavelet=wavelet, tuned=rng.random() < 0.4)
    if kind == "separate":
        return dict(kind=kind, L=rng.choice([128, 256, 512, 1024]), dict=rng.choice(["default", "demo80"]),
                    shift=shift, level2=rng.randint(2, 5), tuned=rng.random() < 0.3)
    if kind == "rdwt":
        levels = rng.randint(1, 5)
        q = 1 << levels
        nimg = rng.randint(1, 6)
        side = math.sqrt(4 * 1000 * 1496 / nimg)
        m = q * max(1, _log(rng, 24, side) // q)
        n = q * max(1, _log(rng, 24, side) // q)
        return dict(kind=kind, nimg=nimg, m=m, n=n, levels=levels, wavelet=wavelet)
    if kind == "mad":
        planes = _log(rng, 1, 200)
        return dict(kind=kind, planes=planes, elems=_log(rng, 500, min(2000000, 49 * 512 * 512 // planes)),
                    arith=rng.choice(["fp64", "fp32"]))
    n, mode = rng.choice([(32, 1.0), (64, 1.0), (128, 1.0), (48, 1.5), (64, 2.0)])
    dirs = rng.choice(["8,8,4", "4,4,4", "6,4,3", "4,3,2"])
    if kind == "bands3d":
        n, mode = (64, 1.0) if n == 128 else (n, mode)
        return dict(kind=kind, n=n, nvol=rng.randint(1, 64 // n), dirs="4,3,2" if dirs == "8,8,4" else dirs, mode=mode)
    return dict(kind=kind, n=n, nvol=rng.randint(1, {128: 2, 64: 6}.get(n, 12)), dirs=dirs, mode=mode)


# ---- inputs ------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _rand(g, *shape, lo=0.0, hi=1.0):
    return lo + (hi - lo) * torch.rand(*shape, generator=g, device=DEV, dtype=F64)


def _images(g, nimg, L):
    """(nimg, L, L) sums of 12 filled ellipses, grey values as in a photograph."""
    r = torch.arange(L, device=DEV, dtype=F64)
    out = torch.zeros(nimg, L, L, device=DEV, dtype=F64)
    s = L / 512.0
    for _ in range(12):
        cy, cx, th = _rand(g, nimg, 1, 1, hi=L), _rand(g, nimg, 1, 1, hi=L), _rand(g, nimg, 1, 1, hi=math.pi)
        a, b = _rand(g, nimg, 1, 1, lo=20 * s, hi=160 * s), _rand(g, nimg, 1, 1, lo=20 * s, hi=160 * s)
        val = _rand(g, nimg, 1, 1, lo=0.0, hi=120.0)
        dy, dx = r[None, :, None] - cy, r[None, None, :] - cx
        u, v = dx * torch.cos(th) + dy * torch.sin(th), -dx * torch.sin(th) + dy * torch.cos(th)
        out += val * ((u / a) ** 2 + (v / b) ** 2 <= 1.0)
    return out


def _noise(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=F64)


def _curves(g, nimg, L):
    """(nimg, L, L) bright strokes along random parabolas."""
    out = torch.zeros(nimg, L, L, device=DEV, dtype=F64)
    r = torch.arange(L, device=DEV, dtype=F64)
    for _ in range(10):
        c0, c1, c2 = (_rand(g, nimg, 1, 1, lo=0.1 * L, hi=0.9 * L), _rand(g, nimg, 1, 1, lo=-1.0, hi=1.0),
                      _rand(g, nimg, 1, 1, lo=-0.5, hi=0.5))
        t = r[None, None, :] - L / 2
        out += 60.0 * ((r[None, :, None] - (c0 + c1 * t + c2 * t * t / L)).abs() < 1.0)
    return out


def _volumes(g, nvol, n):
    r = torch.arange(n, device=DEV, dtype=F64)
    out = torch.zeros(nvol, n, n, n, device=DEV, dtype=F64)
    for _ in range(8):
        c, a = _rand(g, 3, nvol, 1, 1, 1, hi=n), _rand(g, 3, nvol, 1, 1, 1, lo=n / 16, hi=n / 3)
        val = _rand(g, nvol, 1, 1, 1, hi=200.0)
        d = ((r.view(1, n, 1, 1) - c[0]) / a[0]) ** 2 + ((r.view(1, 1, n, 1) - c[1]) / a[1]) ** 2
        out += val * (d + ((r.view(1, 1, 1, n) - c[2]) / a[2]) ** 2 <= 1.0)
    return out


def _gap(mags, t):
    """t moved by at most 5% to the middle of the widest gap of the magnitudes
    around it (a 0-dim tensor)."""
    v = mags.reshape(-1)
    v = v[(v > 0.95 * t) & (v < 1.05 * t)]
    ends = torch.tensor([0.95 * float(t), 1.05 * float(t)], device=v.device, dtype=v.dtype)
    v = torch.sort(torch.cat([v, ends])).values
    i = torch.argmax(v[1:] - v[:-1])
    return 0.5 * (v[i] + v[i + 1])


# ---- the transforms in 64 bits -------------------------------------------------------

class Nsst64:
    """Forward and inverse 2D transform of images (..., L, L), double precision."""

    def __init__(self, L, name, shift):
        self.L = L
        self.dcomp, self.dsize = DICTS[name]
        self.S = len(self.dcomp)
        self.ndir = [1 << c for c in self.dcomp]
        self.H = []
        for w in dictionary_filters(self.dcomp, self.dsize):
            p = torch.zeros(w.shape[0], L, L, dtype=F64, device=DEV)
            p[:, :w.shape[1], :w.shape[2]] = torch.from_numpy(np.ascontiguousarray(w)).to(DEV)
            if shift == "center":
                p = torch.roll(p, (-(w.shape[1] // 2), -(w.shape[2] // 2)), dims=(1, 2))
            h = torch.fft.rfft2(p)
            self.H.append(h / torch.sqrt((h.abs() ** 2).sum(0)))
        self.flt = [torch.from_numpy(np.ascontiguousarray(f)).to(DEV) for f in api.maxflat_filters()]
        imp = torch.zeros(L, L, dtype=F64, device=DEV)
        imp[L // 2, L // 2] = 1.0
        self.norms = [(c.reshape(-1, L * L) ** 2).sum(1).sqrt().cpu().numpy() for c in self.dec(imp)]

    def response(self, which, m):
        """Response of a symmetric filter at dilation m on the 2L-periodic grid."""
        h, n = self.flt[which], 2 * self.L
        at = ((torch.arange(h.shape[0], device=DEV) - h.shape[0] // 2) * m) % n
        k = torch.zeros(n, n, dtype=F64, device=DEV)
        k.index_put_((at[:, None].expand_as(h), at[None, :].expand_as(h)), h, accumulate=True)
        return torch.fft.rfft2(k).real

    def ext(self, x):
        x = torch.cat([x, x.flip(-2)], -2)
        return torch.fft.rfft2(torch.cat([x, x.flip(-1)], -1))

    def crop(self, X):
        return torch.fft.irfft2(X, s=(2 * self.L, 2 * self.L))[..., :self.L, :self.L]

    def pyr_dec(self, x, levels):
        """[lowpass, coarsest ... finest]"""
        X, y = self.ext(x), []
        for lev in range(levels):
            y.insert(0, self.crop(X * self.response(1, 1 << lev)))
            X = X * self.response(0, 1 << lev)
        return [self.crop(X)] + y

    def pyr_rec(self, y):
        levels = len(y) - 1
        X = self.ext(y[0])
        for lev in range(levels - 1, -1, -1):
            X = X * self.response(2, 1 << lev) + self.ext(y[levels - lev]) * self.response(3, 1 << lev)
        return self.crop(X)

    def dec(self, x):
        """[lowpass (..., L, L), scale j (..., D_j, L, L)]"""
        y = self.pyr_dec(x, self.S)
        return [y[0]] + [torch.fft.irfft2(torch.fft.rfft2(v).unsqueeze(-3) * h, s=(self.L, self.L))
                         for v, h in zip(y[1:], self.H)]

    def rec(self, C):
        y = [torch.fft.irfft2((torch.fft.rfft2(c) * h.conj()).sum(-3), s=(self.L, self.L))
             for c, h in zip(C[1:], self.H)]
        return self.pyr_rec([C[0]] + y)

    def flat(self, C):
        """(..., 1 + sum D, L, L)"""
        return torch.cat([C[0].unsqueeze(-3)] + C[1:], -3)

    def cells(self, flat):
        out, k = [flat[..., 0, :, :]], 1
        for d in self.ndir:
            out.append(flat[..., k:k + d, :, :])
            k += d
        return out

    def thresholds(self, flat, sigma, T):
        """Gap-placed T * sigma * norm of every band of one image's (or, over
        the leading axis, all images') coefficients."""
        t = [T[0]] + [T[1] if j < self.S - 1 else T[2] for j, d in enumerate(self.ndir) for _ in range(d)]
        s = np.concatenate(self.norms)
        return [_gap(flat[..., b, :, :].abs(), t[b] * sigma * s[b]) if t[b] else torch.zeros((), device=DEV, dtype=F64)
                for b in range(len(t))]


@functools.lru_cache(maxsize=4)
def _nsst64(L, name, shift):
    return Nsst64(L, name, shift)


def _hard(c, th):
    return torch.where(c.abs() > th, c, torch.zeros_like(c))


def _soft(c, th):
    return torch.sign(c) * torch.clamp(c.abs() - th, min=0)


def _taps(h):
    """Analysis taps (low, high) of the undecimated transform."""
    h = [float(v) for v in h]
    n = len(h)
    return h, [h[n - 1 - j] * (-1.0 if (n - 1 - j) % 2 == 0 else 1.0) for j in range(n)]


def _filt(x, taps, step, dim):
    return sum(t * torch.roll(x, -j * step, dims=dim) for j, t in enumerate(taps))


def mrdwt64(x, h, levels):
    a0, a1 = _taps(h)
    yh = []
    for lev in range(levels):
        A, B = _filt(x, a0, 1 << lev, -1), _filt(x, a1, 1 << lev, -1)
        yh += [_filt(A, a1, 1 << lev, -2), _filt(B, a0, 1 << lev, -2), _filt(B, a1, 1 << lev, -2)]
        x = _filt(A, a0, 1 << lev, -2)
    return x, torch.cat(yh, -1)


def mirdwt64(x, yh, h, levels):
    n, k = x.shape[-1], len(h)
    g0 = [float(v) / 2 for v in h]
    g1 = [float(h[k - 1 - t]) / 2 * (-1.0 if t % 2 else 1.0) for t in range(k)]
    syn = lambda u, v, step, dim: _filt(u, g0, -step, dim) + _filt(v, g1, -step, dim)  # noqa: E731
    for lev in range(levels - 1, -1, -1):
        lh, hl, hh = (yh[..., (3 * lev + i) * n:(3 * lev + i + 1) * n] for i in range(3))
        x = syn(syn(x, lh, 1 << lev, -2), syn(hl, hh, 1 << lev, -2), 1 << lev, -1)
    return x


def _wave_cols(th, n, levels):
    """(3 n levels,) thresholds along a row of yh from 3 * levels band values."""
    return torch.repeat_interleave(th, n)[:3 * n * levels]


def _wave_norms(h, levels):
    x = torch.zeros(256, 256, dtype=F64, device=DEV)
    x[128, 128] = 1.0
    yl, yh = mrdwt64(x, h, levels)
    return [float(yl.norm())] + [float(yh[:, i * 256:(i + 1) * 256].norm()) for i in range(3 * levels)]


class Vol64:
    """The 3D path of volumes (n, n, n), double precision."""

    def __init__(self, n, dirs, mode):
        self.dirs = [int(d) for d in dirs.split(",")]
        self.L, self.n = len(self.dirs), n
        L = self.L
        self.w, self.tb, self.D = {
            1.0: ([0.5] + [0.25] * (L - 1), [1 / 6] + [1 / 12] * (L - 1), [1] + [2] * (L - 1)),
            1.5: ([0.5] + [3 / 8] * (L - 1), [1 / 7] + [1 / 9] * (L - 1), [1.5] + [2] * (L - 1)),
            2.0: ([1 / 3] * L, [1 / 7] * L, [2] * L)}[mode]
        self.sides = [n]
        for d in self.D:
            self.sides.append(int(round(self.sides[-1] / d)))
        self.filt = [torch.from_numpy(np.float32(f)).to(DEV) for f in _cones(dirs)]
        imp = torch.zeros(n, n, n, dtype=F64, device=DEV)
        imp[n // 2, n // 2, n // 2] = 1.0
        subs = self.dec(imp)
        self.norms = [float(b.norm()) * (n / self.sides[l]) ** 1.5 for l in range(L) for b in self.bands(subs, l)]

    def lowpass(self, l):
        """Per-axis passband factor of level l over its FFT frequencies, and its edge."""
        n = self.sides[l]
        P = math.ceil(n / 2 * (self.w[l] + self.tb[l]))
        den = P - math.floor(n / 2 * (self.w[l] - self.tb[l]))
        f = np.abs(np.fft.fftfreq(n, 1.0 / n))
        t = np.clip((P - f) / den, 0.0, 1.0)
        v = torch.from_numpy(np.sqrt(0.5 * (1 - np.cos(np.pi * t)))).to(DEV)
        return v[:, None, None] * v[None, :, None] * v[None, None, :n // 2 + 1], P

    def small(self, l, P):
        """Frequencies of the passband box on the grid of level l and of the next one."""
        n, m = self.sides[l], self.sides[l + 1]
        f = torch.arange(-P, P + 1, device=DEV)
        big, sml, half = f % n, f % m, torch.arange(P + 1, device=DEV)
        return (big[:, None, None], big[None, :, None], half[None, None, :]), (sml[:, None, None], sml[None, :, None],
                                                                              half[None, None, :])

    def irfft(self, X, side):
        return torch.fft.irfftn(X, s=(side,) * 3)

    def dec(self, x):
        X, subs = torch.fft.rfftn(x), []
        for l in range(self.L):
            lf, P = self.lowpass(l)
            subs.append(self.irfft(X * torch.sqrt(1 - lf * lf), self.sides[l]))
            m = self.sides[l + 1]
            big, sml = self.small(l, P)
            Y = torch.zeros(m, m, m // 2 + 1, dtype=torch.complex128, device=DEV)
            Y[sml] = (X * lf)[big] / self.D[l] ** 1.5
            X = Y
        return subs + [self.irfft(X, self.sides[-1])]

    def rec(self, subs):
        X = torch.fft.rfftn(subs[-1])
        for l in range(self.L - 1, -1, -1):
            lf, P = self.lowpass(l)
            big, sml = self.small(l, P)
            Y = torch.fft.rfftn(subs[l]) * torch.sqrt(1 - lf * lf)
            Z = torch.zeros_like(Y)
            Z[big] = X[sml] * self.D[l] ** 1.5
            X = Y + Z * lf
        return self.irfft(X, self.n)

    def grid(self, l):
        return self.sides[l] + 16

    def bands(self, subs, l):
        """The bands of level l one by one: 'same' convolution, offset 12."""
        n, N = self.sides[l], self.grid(l)
        S = torch.fft.rfftn(subs[l], s=(N,) * 3)
        for f in self.filt[l]:
            yield self.irfft(S * torch.fft.rfftn(f.double(), s=(N,) * 3), N)[12:12 + n, 12:12 + n, 12:12 + n]

    def adjoint(self, bands, l):
        n, N = self.sides[l], self.grid(l)
        acc = 0
        for b, f in zip(bands, self.filt[l]):
            p = torch.zeros(N, N, N, dtype=F64, device=DEV)
            p[12:12 + n, 12:12 + n, 12:12 + n] = b
            acc = acc + torch.fft.rfftn(p) * torch.fft.rfftn(f.double(), s=(N,) * 3).conj()
        return self.irfft(acc, N)[:n, :n, :n]


@functools.lru_cache(maxsize=4)
def _cones(dirs):
    return get_meyer_based_filter([int(d) for d in dirs.split(",")])


@functools.lru_cache(maxsize=2)
def _vol64(n, dirs, mode):
    return Vol64(n, dirs, mode)


def _f32(x):
    return x.to(torch.float32).contiguous()


# ---- prepare / run / exact per kind ---------------------------------------------------

def _dictionary(case):
    dcomp, dsize = DICTS[case["dict"]]
    return api.make_dictionary(case["L"], dcomp, dsize, case["shift"])


class Denoise:
    T = (0.0, 3.0, 4.0)

    def inputs(self, c, seed):
        g = _gen(seed)
        L = c["L"]
        x = _f32(_images(g, 1, L)[0] + c["sigma"] * _noise(g, L, L))
        ref = _nsst64(L, c["dict"], c["shift"])
        th = torch.stack(ref.thresholds(ref.flat(ref.dec(x.double())), c["sigma"], self.T)).cpu().numpy()
        # the noise scalars that give these thresholds
        t = [1.0] + [self.T[1] if j < ref.S - 1 else self.T[2] for j, d in enumerate(ref.ndir) for _ in range(d)]
        sc = th / (np.array(t) * c["sigma"])
        cells, k = [float(sc[0])], 1
        for d in ref.ndir:
            cells.append(sc[k:k + d])
            k += d
        return x, th, cells

    def prepare(self, c, seed):
        x, _, sc = self.inputs(c, seed)
        shear = _dictionary(c)
        if c["tuned"]:
            api.autotune(shear)
        Ct = shear.alloc_coeffs() if c["coeffs"] else None
        out = torch.empty_like(x)
        st = dict(c=c, x=x, sc=sc, shear=shear, Ct=Ct, out=out)
        if c["graph"]:
            st["g"] = api.denoise_graph(x, shear, c["sigma"], sc, self.T, Ct=Ct, out=out, coeffs=c["coeffs"])[0]
        return st

    def run(self, st):
        c = st["c"]
        if c["graph"]:
            st["g"].launch()
        else:
            api.denoise_cuda(st["x"], st["shear"], c["sigma"], st["sc"], self.T, Ct=st["Ct"], out=st["out"],
                             coeffs=c["coeffs"])
        return [st["out"]] + (list(st["Ct"]) if c["coeffs"] else [])

    def exact(self, c, seed):
        x, th, _ = self.inputs(c, seed)
        ref = _nsst64(c["L"], c["dict"], c["shift"])
        C = ref.dec(x.double())
        kept = _hard(ref.flat(C), torch.from_numpy(th).to(DEV)[:, None, None])
        return [ref.rec(ref.cells(kept))] + (C if c["coeffs"] else [])


class Transform:
    def inputs(self, c, seed):
        g = _gen(seed)
        return _f32(_images(g, 1, c["L"])[0] + 10.0 * _noise(g, c["L"], c["L"]))

    def prepare(self, c, seed):
        shear = _dictionary(c)
        x = self.inputs(c, seed)
        return dict(c=c, x=x, shear=shear, Ct=shear.alloc_coeffs(), out=torch.empty_like(x))

    def run(self, st):
        Ct = api.shear_trans_cuda(st["x"], "maxflat", st["shear"], st["Ct"])
        return Ct + [api.inverse_shear_cuda(Ct, "maxflat", st["shear"], st["out"])]

    def exact(self, c, seed):
        ref = _nsst64(c["L"], c["dict"], c["shift"])
        C = ref.dec(self.inputs(c, seed).double())
        return C + [ref.rec(C)]


class BatchDenoise:
    T = (0.0, 3.0, 4.0)

    def inputs(self, c, seed):
        g = _gen(seed)
        n, L = c["nimg"], c["L"]
        sig = _rand(g, n, lo=8.0, hi=30.0)
        x = _f32(_images(g, n, L) + sig[:, None, None] * _noise(g, n, L, L))
        ref = _nsst64(L, c["dict"], c["shift"])
        th = torch.stack([torch.stack(ref.thresholds(ref.flat(ref.dec(x[i].double())), s, self.T))
                          for i, s in enumerate(sig.tolist())])
        return x, _f32(th)

    def prepare(self, c, seed):
        x, th = self.inputs(c, seed)
        shear = _dictionary(c)
        b = api.Batch(shear, c["nimg"])
        if c["tuned"]:
            api.autotune(shear, b)
        return dict(c=c, x=x, th=th, shear=shear, b=b, C=b.alloc_coeffs() if c["coeffs"] else None,
                    out=torch.empty_like(x))

    def run(self, st):
        st["b"].denoise(st["x"], st["C"], st["th"], st["out"])
        return [st["out"]] + ([st["C"]] if st["C"] is not None else [])

    def exact(self, c, seed):
        x, th = self.inputs(c, seed)
        ref = _nsst64(c["L"], c["dict"], c["shift"])
        outs, Cs = [], []
        for i in range(c["nimg"]):
            flat = ref.flat(ref.dec(x[i].double()))
            outs.append(ref.rec(ref.cells(_hard(flat, th[i].double()[:, None, None]))))
            if c["coeffs"]:
                Cs.append(flat.cpu())
        return [torch.stack(outs)] + ([torch.stack(Cs)] if c["coeffs"] else [])


class Train:
    """c = S(soft(A x)), p = W^-1(soft(W(x - c))), squared errors of both parts."""

    def inputs(self, c, seed):
        g = _gen(seed)
        n, L, h = c["nimg"], c["L"], MakeONFilter(*WAVELETS[c["wavelet"]])
        cartoon, curves = _images(g, n, L), _curves(g, n, L)
        x = _f32(cartoon + curves + 10.0 * _noise(g, n, L, L))
        ref = _nsst64(L, c["dict"], c["shift"])
        flat = torch.stack([ref.flat(ref.dec(v.double())) for v in x])
        th_sh = _f32(torch.stack(ref.thresholds(flat, 10.0, (3.0, 3.0, 3.0))))
        part = torch.stack([ref.rec(ref.cells(_soft(f, th_sh.double()[:, None, None]))) for f in flat])
        yl, yh = mrdwt64(x.double() - part, h, c["levels"])
        wn = _wave_norms(h, c["levels"])
        th_w = [_gap(yl.abs(), 30.0 * wn[0])]
        th_w += [_gap(yh[..., i * L:(i + 1) * L].abs(), 30.0 * wn[i + 1]) for i in range(3 * c["levels"])]
        return x, _f32(curves), _f32(cartoon), th_sh, _f32(torch.stack(th_w)), h

    def prepare(self, c, seed):
        x, curves, cartoon, th_sh, th_w, h = self.inputs(c, seed)
        shear = _dictionary(c)
        plan = api.Batch(shear, c["nimg"])
        if c["tuned"]:
            api.autotune(shear, plan)
        return dict(c=c, x=x.requires_grad_(True), curves=curves, cartoon=cartoon, h=h, shear=shear, plan=plan,
                    th_sh=th_sh.requires_grad_(True), th_w=th_w.requires_grad_(True))

    def run(self, st):
        part, rest = separation.unrolled_separation(st["x"], st["th_sh"], st["th_w"], st["plan"], st["h"],
                                                    st["c"]["levels"], 1)
        loss = torch.mean((part - st["curves"]) ** 2) + torch.mean((rest - st["cartoon"]) ** 2)
        grads = torch.autograd.grad(loss, [st["x"], st["th_sh"], st["th_w"]])
        return [part.detach(), rest.detach()] + list(grads)

    def exact(self, c, seed):
        x, curves, cartoon, th_sh, th_w, h = self.inputs(c, seed)
        ref = _nsst64(c["L"], c["dict"], c["shift"])
        th_sh, th_w = th_sh.double().requires_grad_(True), th_w.double().requires_grad_(True)
        outs, gx, gs, gw = [], [], 0, 0
        for i in range(c["nimg"]):  # one image at a time: the losses and threshold gradients add up
            v = x[i].double().requires_grad_(True)
            part = ref.rec(ref.cells(_soft(ref.flat(ref.dec(v)), th_sh[:, None, None])))
            yl, yh = mrdwt64(v - part, h, c["levels"])
            rest = mirdwt64(_soft(yl, th_w[0]), _soft(yh, _wave_cols(th_w[1:], c["L"], c["levels"])), h, c["levels"])
            loss = (torch.mean((part - curves[i].double()) ** 2) +
                    torch.mean((rest - cartoon[i].double()) ** 2)) / c["nimg"]
            a, b, d = torch.autograd.grad(loss, [v, th_sh, th_w])
            outs.append((part.detach(), rest.detach()))
            gx.append(a)
            gs, gw = gs + b, gw + d
        return [torch.stack([o[0] for o in outs]), torch.stack([o[1] for o in outs]), torch.stack(gx), gs, gw]


class Separate:
    WEIGHTS = [0.1, 0.1, 1.5, 1.5]
    DELTA, GAMMA = 30.0, 3.0

    def steps64(self, c, img, p1, p2, th=None, tw=None):
        """One iteration in 64 bits; without thresholds, the gap-placed ones."""
        ref = _nsst64(c["L"], c["dict"], c["shift"])
        y = ref.pyr_dec(img, len(self.WEIGHTS) - 1)
        x = ref.pyr_rec([w * v for w, v in zip(self.WEIGHTS, y)])
        r = x - p1 - p2
        flat = ref.flat(ref.dec(p1 + r))
        h, haar = MakeONFilter("Symmlet", 4), MakeONFilter("Haar")
        yl, yh = mrdwt64(p2 + r, h, c["level2"])
        if th is None:
            s = np.concatenate(ref.norms)
            th = torch.stack([_gap(flat[b].abs(), self.DELTA * s[b]) for b in range(len(s))])
            tw = _gap(yh.abs(), self.DELTA)
            return th, tw
        a = ref.rec(ref.cells(_hard(flat, th[:, None, None])))
        ll, wc = mrdwt64(a, haar, 1)
        return [mirdwt64(ll, _soft(wc, self.GAMMA), haar, 1), mirdwt64(yl, _hard(yh, tw), h, c["level2"])]

    def inputs(self, c, seed):
        g = _gen(seed)
        L = c["L"]
        cartoon, curves = _images(g, 1, L)[0], _curves(g, 1, L)[0]
        img = _f32(cartoon + curves + 10.0 * _noise(g, L, L))
        p1, p2 = _f32(0.6 * curves), _f32(0.4 * cartoon)
        th, tw = self.steps64(c, img.double(), p1.double(), p2.double())
        return img, p1, p2, _f32(th), float(_f32(tw))

    def prepare(self, c, seed):
        img, p1, p2, th, tw = self.inputs(c, seed)
        shear = _dictionary(c)
        if c["tuned"]:
            api.autotune(shear)
        # thresh_cuda takes lambda * E(cell, direction): the thresholds as norms
        E, v, k = np.zeros((shear.nscales + 1, max(shear.ndir))), th.double().cpu().numpy(), 0
        for j, d in enumerate([1] + shear.ndir):
            E[j, :d] = v[k:k + d]
            k += d
        return dict(c=c, img=img, p1=p1, p2=p2, E=E, tw=tw, shear=shear, ones=np.ones(shear.nscales + 1),
                    Ct=shear.alloc_coeffs(), h=MakeONFilter("Symmlet", 4), haar=MakeONFilter("Haar"))

    def run(self, st):
        c, shear, Ct = st["c"], st["shear"], st["Ct"]
        x = api.re_weight_band_cuda(st["img"], self.WEIGHTS, shear)
        r = x - st["p1"] - st["p2"]
        api.shear_trans_cuda(st["p1"] + r, "maxflat", shear, Ct)
        api.thresh_cuda(Ct, 1.0, 2, st["E"], st["ones"], 0)
        a = separation.tv_correction_cuda(api.inverse_shear_cuda(Ct, "maxflat", shear), self.GAMMA, st["haar"])
        yl, yh = api.mrdwt_cuda(st["p2"] + r, st["h"], c["level2"])
        api.thresh_cuda([yl, yh], st["tw"], 1, st["E"], np.zeros(1), 0)
        return [a, api.mirdwt_cuda(yl, yh, st["h"], c["level2"])]

    def exact(self, c, seed):
        img, p1, p2, th, tw = self.inputs(c, seed)
        return self.steps64(c, img.double(), p1.double(), p2.double(), th.double(), tw)


class Rdwt:
    def inputs(self, c, seed):
        g = _gen(seed)
        s = (c["nimg"], c["m"], c["n"])
        smooth = torch.cumsum(_noise(g, *s), -1) * 2.0
        return _f32(128.0 + smooth - smooth.mean(-1, keepdim=True) + 10.0 * _noise(g, *s))

    def prepare(self, c, seed):
        return dict(c=c, x=self.inputs(c, seed), h=MakeONFilter(*WAVELETS[c["wavelet"]]))

    def run(self, st):
        yl, yh = api.mrdwt_cuda(st["x"], st["h"], st["c"]["levels"])
        return [yl, yh, api.mirdwt_cuda(yl, yh, st["h"], st["c"]["levels"])]

    def exact(self, c, seed):
        h = MakeONFilter(*WAVELETS[c["wavelet"]])
        yl, yh = mrdwt64(self.inputs(c, seed).double(), h, c["levels"])
        return [yl, yh, mirdwt64(yl, yh, h, c["levels"])]


class Mad:
    def inputs(self, c, seed):
        g = _gen(seed)
        s = torch.exp(_rand(g, c["planes"], 1, lo=-4.0, hi=1.0))
        return _f32(s * _noise(g, c["planes"], c["elems"]))

    def prepare(self, c, seed):
        return dict(c=c, x=self.inputs(c, seed))

    def run(self, st):
        return api.band_mad_cuda(st["x"], st["c"]["arith"])

    def exact(self, c, seed):
        def median(v):
            v = torch.sort(v, -1).values
            k = v.shape[-1]
            return (v[..., (k - 1) // 2] + v[..., k // 2]) / 2
        x = self.inputs(c, seed)
        x = x.double() if c["arith"] == "fp64" else x
        return torch.stack([median((v - median(v)).abs()).double() / 0.6745 for v in x])


class Volume:
    T, SIGMA = 3.0, 25.0

    def inputs(self, c, seed):
        g = _gen(seed)
        n = c["n"]
        x = _f32(_volumes(g, c["nvol"], n) + self.SIGMA * _noise(g, c["nvol"], n, n, n))
        ref, th = _vol64(n, c["dirs"], c["mode"]), []
        for v in x:
            subs = ref.dec(v.double())
            bands = (b for l in range(ref.L) for b in ref.bands(subs, l))
            th.append(torch.stack([_gap(b.abs(), self.T * self.SIGMA * s) for b, s in zip(bands, ref.norms)]))
        return x, _f32(torch.stack(th))

    def prepare(self, c, seed):
        x, th = self.inputs(c, seed)
        sh = shearlet3d.Shear3D(c["n"], [int(d) for d in c["dirs"].split(",")], c["mode"], _cones(c["dirs"]))
        return dict(c=c, x=x, th=th, sh=sh, plan=shearlet3d.Plan3D(sh, c["nvol"]), out=torch.empty_like(x))

    def run(self, st):
        return st["plan"].denoise(st["x"], st["th"], st["out"])

    def exact(self, c, seed):
        x, th = self.inputs(c, seed)
        ref, out = _vol64(c["n"], c["dirs"], c["mode"]), []
        for v, t in zip(x, th.double()):
            subs, k = ref.dec(v.double()), 0
            rec = []
            for l in range(ref.L):
                acc = 0
                for b in ref.bands(subs, l):
                    acc = acc + _hard(b, t[k])
                    k += 1
                rec.append(acc)
            out.append(ref.rec(rec + [subs[-1]]))
        return torch.stack(out)


class Bands3d:
    def inputs(self, c, seed):
        g = _gen(seed)
        n = c["n"]
        return _f32(_volumes(g, c["nvol"], n) + 25.0 * _noise(g, c["nvol"], n, n, n))

    def prepare(self, c, seed):
        sh = shearlet3d.Shear3D(c["n"], [int(d) for d in c["dirs"].split(",")], c["mode"], _cones(c["dirs"]))
        plan = shearlet3d.Plan3D(sh, c["nvol"])
        x = self.inputs(c, seed)
        return dict(c=c, x=x, sh=sh, plan=plan, subs=plan.new_subs(), bands=plan.new_bands(), bar=plan.new_subs(),
                    out=torch.empty_like(x))

    def run(self, st):
        p = st["plan"]
        subs = p.pyr_dec(st["x"], st["subs"])
        bands = p.analysis(subs, st["bands"])
        return [subs, bands, p.analysis_adjoint(bands, st["bar"]), p.pyr_rec(subs, st["out"])]

    def exact(self, c, seed):
        ref = _vol64(c["n"], c["dirs"], c["mode"])
        S, B, A, R = [], [], [], []
        for v in self.inputs(c, seed):
            subs = ref.dec(v.double())
            lev = [torch.stack(list(ref.bands(subs, l))) for l in range(ref.L)]
            S.append(torch.cat([s.reshape(-1) for s in subs]))
            B.append(torch.cat([b.reshape(-1) for b in lev]))
            adj = [ref.adjoint(lev[l], l).reshape(-1) for l in range(ref.L)]
            A.append(torch.cat(adj + [torch.zeros_like(subs[-1].reshape(-1))]))  # the lowpass slot is not written
            R.append(ref.rec(subs))
        return [torch.stack(v) for v in (S, B, A, R)]


KINDS = {"denoise": Denoise(), "transform": Transform(), "batch": BatchDenoise(), "train": Train(),
         "separate": Separate(), "rdwt": Rdwt(), "mad": Mad(), "volume": Volume(), "bands3d": Bands3d()}


def prepare(case, seed):
    return KINDS[case["kind"]].prepare(case, seed)


def run(state):
    return KINDS[state["c"]["kind"]].run(state)


def exact(case, seed):
    with torch.no_grad() if case["kind"] != "train" else torch.enable_grad():
        return KINDS[case["kind"]].exact(case, seed)


# ---- what a pass cannot do without ---------------------------------------------------

def _fft2(L):
    """Flops of a real 2D FFT of L x L."""
    return 2.5 * L * L * math.log2(L * L)


def _nsst_work(L, name):
    """(bands, distinct filter bytes, flops of one direction of the transform)."""
    dcomp, dsize = DICTS[name]
    nb, S = sum(1 << d for d in dcomp), len(dcomp)
    filt = sum(1 << d for d, _ in set(zip(dcomp, dsize)))
    return nb, 4.0 * L * L * filt, (nb + 2 * S + 2) * _fft2(L) + 3.0 * L * L * nb


def work(case):
    k = case["kind"]
    if k in ("denoise", "transform", "batch", "train", "separate"):
        L = case["L"]
        P, n = 4.0 * L * L, case.get("nimg", 1)
        nb, filt, fl = _nsst_work(L, case["dict"])
        if k == "denoise" or k == "batch":
            return {"bytes": filt + n * P * (2 + (1 + nb if case["coeffs"] else 0)), "flops": 2 * n * fl}
        if k == "transform":
            return {"bytes": 2 * filt + P * (2 + 2 * (1 + nb)), "flops": 2 * fl}
        taps = len(MakeONFilter(*WAVELETS[case.get("wavelet", "sym4")]))
        lev = case.get("levels", case.get("level2"))
        wav = 2 * 12.0 * taps * lev * L * L
        if k == "train":  # x, both targets in; both parts and x's gradient out; the pass back costs as much
            return {"bytes": 2 * filt + n * P * 6, "flops": n * (4 * fl + 2 * wav)}
        return {"bytes": filt + P * 5, "flops": 2 * fl + wav}
    if k == "rdwt":
        px, taps = case["nimg"] * case["m"] * case["n"], len(MakeONFilter(*WAVELETS[case["wavelet"]]))
        # x in, the bands out; the bands in, x out
        return {"bytes": 4.0 * px * 2 * (2 + 3 * case["levels"]), "flops": 2 * 12.0 * taps * case["levels"] * px}
    if k == "mad":
        return {"bytes": 4.0 * case["planes"] * case["elems"], "flops": 2.0 * case["planes"] * case["elems"]}
    n, dirs = case["n"], [int(d) for d in case["dirs"].split(",")]
    D = {1.0: [1, 2, 2], 1.5: [1.5, 2, 2], 2.0: [2, 2, 2]}[case["mode"]]
    byts, flops, side, grids = 8.0 * n ** 3, 0.0, float(n), set()
    bands = 0.0
    for l, d in enumerate(dirs):
        nb, N = 3 * d * d, side + 12
        if (d, N) not in grids:  # half spectra of the filters, shared by levels of one grid
            grids.add((d, N))
            byts += 4.0 * N ** 3 * nb / case["nvol"]
        flops += (nb + 3) * 2.5 * N ** 3 * 3 * math.log2(N) + 6.0 * nb * N ** 3 / 2
        bands += 4.0 * nb * side ** 3
        side /= D[l]
    if k == "bands3d":
        byts, flops = byts + 2 * bands + 12.0 * n ** 3, 2 * flops
    return {"bytes": case["nvol"] * byts, "flops": case["nvol"] * flops}
