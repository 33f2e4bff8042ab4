"""Device median absolute deviation (shx_band_mad, shx_nsst_scalars) against
numpy's median on the same FP32 data, bit for bit.

numpy's median is the library routine both conventions reduce to:
  fp64  values widened to double, m = median(v), MAD = median(|v - m|) / 0.6745
        (nsst_scalars.m:36-44 on a double transform);
  fp32  the same in float arithmetic (numpy's float32 median averages the two
        middle values in float32, as demo_denoise/shearcuda/shearcuda.cpp:165-181
        does), the final division in double.
Cases cover odd and even counts, one and two elements, ties around the middle,
constant planes, signed zeros, tiny values and both load paths (plane stride a
multiple of four or not).
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _mad64(v):
    v = np.asarray(v, dtype=np.float32).astype(np.float64).ravel()
    return np.median(np.abs(v - np.median(v))) / 0.6745


def _mad32(v):
    v = np.asarray(v, dtype=np.float32).ravel()
    m = np.median(v)
    return float(np.median(np.abs(v - m))) / 0.6745


def _planes(n, kind, nplanes, seed):
    rng = np.random.default_rng(seed)
    if kind == "normal":
        a = rng.standard_normal((nplanes, n)) * 3.0
    elif kind == "ties":
        a = np.round(rng.standard_normal((nplanes, n)) * 2.0)
    elif kind == "const":
        a = np.full((nplanes, n), -1.25)
    elif kind == "zeros":
        a = np.where(rng.random((nplanes, n)) < 0.5, -0.0, 0.0)
    elif kind == "tiny":
        a = rng.standard_normal((nplanes, n)) * 1e-30
    else:  # wide: magnitudes over many binades, both signs
        a = rng.standard_normal((nplanes, n)) * 10.0 ** rng.integers(-20, 20, (nplanes, n))
    return a.astype(np.float32)


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 63, 64, 1001, 4096, 65539, 262144])
@pytest.mark.parametrize("kind", ["normal", "ties", "const", "zeros", "tiny", "wide"])
def test_band_mad_matches_numpy(gpu, n, kind):
    from shearcuda_amd import api
    nplanes = 3 if n < 100000 else 2
    a = _planes(n, kind, nplanes, n * 7 + len(kind))
    t = torch.from_numpy(a).cuda()
    for arith, ref in (("fp64", _mad64), ("fp32", _mad32)):
        got = api.band_mad_cuda(t, arith).cpu().numpy()
        want = np.array([ref(a[i]) for i in range(nplanes)])
        assert np.array_equal(got, want), (n, kind, arith, got, want)


def test_band_mad_unaligned_planes(gpu):
    """A stack whose planes start off 16-byte boundaries (odd plane length)
    and a view that starts one element into its allocation."""
    from shearcuda_amd import api
    a = _planes(4097, "normal", 5, 3)
    base = torch.from_numpy(np.concatenate([[0.0], a.ravel()]).astype(np.float32)).cuda()
    t = base[1:].view(5, 4097)
    got = api.band_mad_cuda(t).cpu().numpy()
    assert np.array_equal(got, np.array([_mad64(r) for r in a]))


@pytest.mark.parametrize("L", [64, 256, 512, 1024])
def test_nsst_scalars_on_device(gpu, L):
    """shx_nsst_scalars: the transform of the noise image, then exact medians,
    equal to numpy on the same coefficients; close to the FP64 oracle's."""
    from oracle import nsst as o
    from shearcuda_amd import api
    from shearcuda_amd.synth import white_noise
    print("case nsst scalars L=%d" % L, flush=True)
    shear = api.make_dictionary(L)
    try:
        w = white_noise(L)
        wg = torch.from_numpy(w.astype(np.float32)).cuda()
        C = api.shear_trans_cuda(wg, "maxflat", shear)
        cells = [C[0].cpu().numpy()[None]] + [c.cpu().numpy() for c in C[1:]]
        for arith, ref in (("fp64", _mad64), ("fp32", _mad32)):
            sc = api.nsst_scalars_cuda(shear, wg, arith)
            got = np.concatenate([[sc[0]]] + [np.asarray(s) for s in sc[1:]])
            want = np.array([ref(p) for c in cells for p in c])
            assert np.array_equal(got, want), arith
        if L == 256:
            so = o.nsst_scalars(o.make_dictionary(L), w)
            ref = np.concatenate([[so[0]]] + [np.asarray(s) for s in so[1:]])
            sc = api.nsst_scalars_cuda(shear, wg)
            got = np.concatenate([[sc[0]]] + [np.asarray(s) for s in sc[1:]])
            err = np.abs(got / ref - 1).max()
            print("L=%d device scalars vs FP64 oracle: max rel %.2e" % (L, err), flush=True)
            assert err < 1e-5
    finally:
        shear.close()


def test_wavelet_scalars_on_device(gpu):
    from oracle import rdwt as w
    from shearcuda_amd import api, separation
    L, levels = 128, 3
    h = w.make_on_filter("Daubechies", 4)
    noise = torch.from_numpy(np.random.default_rng(2).standard_normal((L, L)).astype(np.float32)).cuda()
    got = separation.wavelet_scalars(noise, h, levels)
    yl, yh = api.mrdwt_cuda(noise, h, levels)
    yl, yh = yl.cpu().numpy(), yh.cpu().numpy().reshape(L, 3 * levels, L)
    want = np.array([_mad64(yl)] + [_mad64(yh[:, k, :]) for k in range(3 * levels)])
    assert np.array_equal(got, want)


def test_scalars_3d_on_device(gpu):
    from shearcuda_amd import shearlet3d
    n = 32
    sh = shearlet3d.Shear3D(n, (8, 8, 4), 1)
    noise = torch.from_numpy(np.random.default_rng(5).standard_normal((n, n, n)).astype(np.float32)).cuda()
    est, low = shearlet3d.nsst_scalars_3d(sh, noise)
    plan = shearlet3d.Plan3D(sh, 1, group=8)
    try:
        subs = plan.pyr_dec(noise.reshape(1, n, n, n).contiguous())
        bands = plan.analysis(subs)
        want = [_mad64(b) for lvl in sh.split_bands(bands) for b in lvl[0].cpu().numpy()]
        want_low = _mad64(sh.split_subs(subs)[-1][0].cpu().numpy())
    finally:
        plan.close()
    assert np.array_equal(est, np.array(want))
    assert low == want_low


@pytest.mark.parametrize("n", [32767, 32768, 32769, 49153, 262147])
@pytest.mark.parametrize("kind", ["offset", "grid", "halves", "spike", "normal"])
def test_band_mad_split_planes(gpu, n, kind):
    """Around the size from which a plane is split over several workgroups:
    values whose middle bin overflows the first histogram (a narrow band of
    values on an offset), equal values beyond the candidate buffer (an integer
    grid; two halves, where the middle pair straddles two bins), and a bin of
    more distinct values than the buffer holds (a dense spike)."""
    from shearcuda_amd import api
    rng = np.random.default_rng(n)
    a = rng.standard_normal((3, n))
    if kind == "offset":
        a = 140.0 + a
    elif kind == "grid":
        a = np.round(a * 2)
    elif kind == "halves":
        a = np.where(np.arange(n) % 2 == 0, -2.0, 1.0) * np.ones((3, 1))
    elif kind == "spike":  # 4096 consecutive floats share the leading 12 bits of their keys
        a = np.float32(1.0) + np.float32(2.0 ** -23) * rng.integers(0, 4096, (3, n)).astype(np.float32)
    a = a.astype(np.float32)
    t = torch.from_numpy(a).cuda()
    for arith, ref in (("fp64", _mad64), ("fp32", _mad32)):
        got = api.band_mad_cuda(t, arith).cpu().numpy()
        want = np.array([ref(r) for r in a])
        assert np.array_equal(got, want), (arith, got, want)


def _best_ms(api, x, reps=20):
    api.band_mad_cuda(x)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    best = float("inf")
    for _ in range(reps):
        ev[0].record()
        api.band_mad_cuda(x)
        ev[1].record()
        torch.cuda.synchronize()
        best = min(best, ev[0].elapsed_time(ev[1]))
    return best


def test_band_mad_time_is_linear_in_the_plane(gpu):
    """One plane of normal values, whose middle bin needs the second histogram,
    four times as large: about four times the time (every pass is linear),
    where a sum over the plane's histograms in every block made it eleven."""
    from shearcuda_amd import api
    gen = torch.Generator("cuda").manual_seed(3)
    ms = {e: _best_ms(api, torch.randn(1, 1 << e, device="cuda", generator=gen), 10) for e in (24, 26)}
    print("MAD of 2^24 and 2^26 elements: %.3f and %.3f ms" % (ms[24], ms[26]), flush=True)
    assert ms[26] < 7 * ms[24]


def test_band_mad_small_planes_two_blocks_to_a_cu(gpu):
    """1, 8 and 16 planes of 4096 for every CU: with room for two blocks on a CU
    a further plane for every CU takes about half of what the first takes (0.43
    to 0.52 measured); a block that fills its CU (a copy of the plane in LDS)
    took 0.74 to 0.86."""
    from shearcuda_amd import api
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    gen = torch.Generator("cuda").manual_seed(4)
    t = {k: _best_ms(api, torch.randn(k * cus, 4096, device="cuda", generator=gen), 40) for k in (1, 8, 16)}
    print("MAD of 1, 8, 16 planes of 4096 per CU: %s ms" % t, flush=True)
    assert t[16] - t[8] < 0.65 * 8 * t[1]


@pytest.mark.parametrize("nplanes,n", [(2, 262145), (8, 819200), (8, 819201), (4, 1 << 20), (5, 1 << 20)])
@pytest.mark.parametrize("kind", ["offset", "normal"])
def test_band_mad_second_bin_forms(gpu, nplanes, n, kind):
    """Both places that find the bin of the second histogram (a launch of its
    own, every block of the gather), on both sides of their rule, with planes
    that need it and planes that do not in one call."""
    from shearcuda_amd import api
    a = np.random.default_rng(n + nplanes).standard_normal((nplanes, n))
    if kind == "offset":  # the first plane needs it for its values too
        a[0] += 140.0
    a = a.astype(np.float32)
    t = torch.from_numpy(a).cuda()
    for arith, ref in (("fp64", _mad64), ("fp32", _mad32)):
        got = api.band_mad_cuda(t, arith).cpu().numpy()
        assert np.array_equal(got, np.array([ref(r) for r in a])), arith


def test_band_mad_of_the_largest_plane(gpu):
    """2^31 - 1 elements, the largest plane the entry point takes: 24-bit whole
    numbers in a scrambled order, each 128 times but one, so both medians are
    known exactly.  Block counts, index steps past the end and workspace
    offsets have to hold in their types; the many equal values send both
    selections through the plane itself."""
    from shearcuda_amd import api
    n, a, chunk = (1 << 31) - 1, 1103515245, 1 << 27   # a odd: i -> a i mod 2^31 is a permutation
    t = torch.empty(1, n, device="cuda")
    for c in range(0, n, chunk):
        i = torch.arange(c, min(n, c + chunk), device="cuda")
        t[0, c:c + chunk] = ((i * a) & ((1 << 31) - 1)) >> 7
    del i
    count = np.full(1 << 24, 128, dtype=np.int64)
    count[(((1 << 31) - 1) * a % (1 << 31)) >> 7] -= 1   # the index the plane stops short of
    mid = (n - 1) // 2
    m = int(np.searchsorted(np.cumsum(count), mid, side="right"))
    dev = np.bincount(np.abs(np.arange(1 << 24) - m), weights=count).astype(np.int64)
    want = int(np.searchsorted(np.cumsum(dev), mid, side="right")) / 0.6745
    print("case largest plane", flush=True)
    assert float(api.band_mad_cuda(t, "fp32")[0]) == want


@pytest.mark.parametrize("nplanes,n", [(64, 49151), (64, 49152), (65, 49152), (65, 98303), (65, 98304), (511, 49152),
                                       (512, 49152), (4096, 32769), (4097, 32769)])
def test_band_mad_around_the_split_rule(gpu, nplanes, n):
    """Plane counts and sizes on both sides of the rule that splits planes over
    blocks: every tenth plane and the last against numpy."""
    from shearcuda_amd import api
    a = np.random.default_rng(n + nplanes).standard_normal((nplanes, n), dtype=np.float32)
    t = torch.from_numpy(a).cuda()
    some = sorted(set(range(0, nplanes, max(1, nplanes // 10))) | {nplanes - 1})
    for arith, ref in (("fp64", _mad64), ("fp32", _mad32)):
        got = api.band_mad_cuda(t, arith).cpu().numpy()[some]
        assert np.array_equal(got, np.array([ref(a[i]) for i in some])), arith


def test_band_mad_in_groups(gpu):
    """More planes than go through the split passes together (2048), the groups
    after the first in the workspace of the ones before: every plane the same
    whichever group it falls in, a few against numpy."""
    from shearcuda_amd import api
    n, nplanes = 49155, 2051
    a = np.random.default_rng(8).standard_normal((7, n), dtype=np.float32)
    t = torch.from_numpy(a).cuda().repeat(293, 1)
    assert t.shape[0] == nplanes
    t[5::7] *= torch.arange(1, 294, device="cuda", dtype=torch.float32)[:, None]
    for arith, ref in (("fp64", _mad64), ("fp32", _mad32)):
        got = api.band_mad_cuda(t, arith).cpu().numpy()
        for k in (0, 1, 2, 3, 4, 6):
            assert np.all(got[k::7] == ref(a[k])), (arith, k)
        for i in (5, 5 + 7 * 146, 5 + 7 * 292):
            assert got[i] == ref(t[i].cpu().numpy()), (arith, i)
