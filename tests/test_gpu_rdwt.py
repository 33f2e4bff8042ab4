"""GPU parity of the undecimated wavelet transform and its adjoints."""
import numpy as np
import pytest
import torch

from oracle import rdwt as w

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api(gpu):
    from shearcuda_amd import api
    return api


def g(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).cuda()


def relmax(a, b):
    return np.abs(np.asarray(a, np.float64) - b).max() / np.abs(b).max()


@pytest.mark.parametrize("name,par,L,shape", [("Daubechies", 4, 3, (512, 512)), ("Symmlet", 4, 2, (64, 128)),
                                              ("Haar", 0, 1, (32, 32))])
def test_mrdwt_mirdwt_match_oracle(api, name, par, L, shape):
    print("case rdwt", name, L, shape, flush=True)
    h = w.make_on_filter(name, par)
    x = np.random.default_rng(L).standard_normal(shape) * 50
    yl, yh = api.mrdwt_cuda(g(x), h, L)
    ryl, ryh = w.mrdwt(x, h, L)
    assert relmax(yl.cpu().numpy(), ryl) < 1e-5
    for lev in range(L):
        for q in range(3):
            c0 = (3 * lev + q) * shape[1]
            assert relmax(yh.cpu().numpy()[:, c0:c0 + shape[1]], ryh[:, c0:c0 + shape[1]]) < 1e-5
    xr = api.mirdwt_cuda(g(ryl), g(ryh), h, L).cpu().numpy()
    assert relmax(xr, w.mirdwt(ryl, ryh, h, L)) < 1e-5


def test_rdwt_batched_equals_single(api):
    h = w.make_on_filter("Daubechies", 4)
    xs = np.random.default_rng(3).standard_normal((3, 64, 64))
    yl, yh = api.mrdwt_cuda(g(xs), h, 3)
    for i in range(3):
        a, b = api.mrdwt_cuda(g(xs[i]), h, 3)
        assert torch.equal(a, yl[i]) and torch.equal(b, yh[i])


def test_rdwt_adjoints_dense(api):
    """Dense matrices of mrdwt / mirdwt on 16x16 (3 levels) from the oracle;
    the adjoint kernels must apply their transposes."""
    print("case rdwt dense adjoint", flush=True)
    h = w.make_on_filter("Daubechies", 4)
    m = n = 16
    L = 3
    N = m * n
    A = np.zeros((N + 3 * N * L, N))   # analysis matrix, rows (yl, yh)
    for i in range(N):
        e = np.zeros(N)
        e[i] = 1
        yl, yh = w.mrdwt(e.reshape(m, n), h, L)
        A[:, i] = np.concatenate([yl.ravel(), yh.ravel()])
    S = np.zeros((N, N + 3 * N * L))   # synthesis matrix
    for i in range(N + 3 * N * L):
        e = np.zeros(N + 3 * N * L)
        e[i] = 1
        S[:, i] = w.mirdwt(e[:N].reshape(m, n), e[N:].reshape(m, 3 * n * L), h, L).ravel()
    rng = np.random.default_rng(7)
    # batch of probes: adjoint of analysis
    P = rng.standard_normal((8, N + 3 * N * L))
    xb = api.mrdwt_adjoint_cuda(g(P[:, :N].reshape(8, m, n)), g(P[:, N:].reshape(8, m, 3 * n * L)), h, L)
    ref = P @ A                      # rows: A^T p
    assert relmax(xb.cpu().numpy().reshape(8, N), ref) < 1e-5
    Q = rng.standard_normal((8, N))
    ylb, yhb = api.mirdwt_adjoint_cuda(g(Q.reshape(8, m, n)), h, L)
    got = np.concatenate([ylb.cpu().numpy().reshape(8, N), yhb.cpu().numpy().reshape(8, -1)], axis=1)
    assert relmax(got, Q @ S) < 1e-5


@pytest.mark.parametrize("name,par", [("Haar", 0), ("Daubechies", 4), ("Daubechies", 6), ("Symmlet", 4)])
@pytest.mark.parametrize("shape,L", [((8, 8), 3), ((32, 64), 5), ((20, 516), 2), ((36, 1044), 2), ((6, 510), 1),
                                     ((64, 1536), 5), ((144, 96), 4)])
def test_rdwt_ragged_shapes(api, name, par, shape, L):
    """Sides around the level kernels' tiles: rows of at most 512 columns in
    one block and longer ones split, strips that end inside a tile, dilations
    longer than the image, every filter length."""
    from shearcuda_amd.wavelets import MakeONFilter
    h = MakeONFilter(name, par)
    x = np.random.default_rng(L).standard_normal((2,) + shape) * 50
    yl, yh = api.mrdwt_cuda(g(x), h, L)
    xr = api.mirdwt_cuda(yl, yh, h, L).cpu().numpy()
    for i in range(2):
        ryl, ryh = w.mrdwt(x[i], h, L)
        assert relmax(yl[i].cpu().numpy(), ryl) < 1e-5
        assert relmax(yh[i].cpu().numpy(), ryh) < 1e-5
        assert relmax(xr[i], x[i]) < 1e-5


# shapes whose strips take 16, 8 and 4 rows (as many as leave 1024 blocks), with rows
# per phase that are no multiple of them; rows of up to 512 columns and longer ones
STRIPS = [(210, 72, 24, 2), (208, 68, 512, 1), (256, 24, 520, 1), (128, 68, 40, 2), (130, 44, 516, 2)]


@pytest.mark.parametrize("name,par", [("Haar", 0), ("Daubechies", 4), ("Daubechies", 6), ("Symmlet", 4)])
@pytest.mark.parametrize("nimg,m,n,L", STRIPS)
def test_rdwt_strips_of_16_and_8_rows(api, name, par, nimg, m, n, L):
    """Strips of 16 and 8 rows (large batches) against the same images in
    batches of four, which take strips of 4: the same sums in the same order,
    so the same bits, for both transforms and both adjoints; two images
    against the oracle."""
    from shearcuda_amd.wavelets import MakeONFilter
    h = MakeONFilter(name, par)
    gen = torch.Generator("cuda").manual_seed(nimg + m)
    x = torch.randn(nimg, m, n, device="cuda", generator=gen) * 50
    yl, yh = api.mrdwt_cuda(x, h, L)
    xr = api.mirdwt_cuda(yl, yh, h, L)
    xa = api.mrdwt_adjoint_cuda(yl, yh, h, L)
    al, ah = api.mirdwt_adjoint_cuda(x, h, L)
    for i in range(0, nimg, 4):
        s = slice(i, min(nimg, i + 4))
        l4, h4 = api.mrdwt_cuda(x[s].contiguous(), h, L)
        assert torch.equal(l4, yl[s]) and torch.equal(h4, yh[s])
        assert torch.equal(api.mirdwt_cuda(l4, h4, h, L), xr[s])
        assert torch.equal(api.mrdwt_adjoint_cuda(l4, h4, h, L), xa[s])
        l4, h4 = api.mirdwt_adjoint_cuda(x[s].contiguous(), h, L)
        assert torch.equal(l4, al[s]) and torch.equal(h4, ah[s])
    for i in (0, nimg - 1):
        ryl, ryh = w.mrdwt(x[i].cpu().numpy(), h, L)
        assert relmax(yl[i].cpu().numpy(), ryl) < 1e-5
        assert relmax(yh[i].cpu().numpy(), ryh) < 1e-5
        assert relmax(xr[i].cpu().numpy(), x[i].cpu().numpy()) < 1e-5


@pytest.mark.parametrize("taps,shape,L", [(10, (24, 40), 2), (12, (36, 1044), 1), (16, (40, 24), 3), (32, (64, 64), 2),
                                          (8, (128, 1024), 7), (6, (64, 576), 6)])
def test_rdwt_separate_passes(api, taps, shape, L):
    """Filters of more than 8 taps and deep levels of long rows, which run as
    separate row and column passes: both transforms against the oracle, both
    adjoints by their identity with the oracle's transforms.  The taps are
    random (the passes do not assume an orthonormal filter)."""
    from shearcuda_amd._lib import lib
    m, n = shape
    fused = lib.shx_rdwt_fused(n, L, taps)
    assert fused == (1 if taps == 6 else 0)   # the last: just inside the fused rule
    rng = np.random.default_rng(taps + L)
    h = rng.standard_normal(taps)
    h /= np.linalg.norm(h)
    x, y = rng.standard_normal((2, 2, m, n)) * 50, rng.standard_normal((2, m, 3 * n * L))
    yl, yh = api.mrdwt_cuda(g(x[0]), h, L)
    back = api.mirdwt_cuda(g(x[0]), g(y), h, L).cpu().numpy()
    xa = api.mrdwt_adjoint_cuda(g(x[0]), g(y), h, L).cpu().numpy().astype(np.float64)
    al, ah = (t.cpu().numpy().astype(np.float64) for t in api.mirdwt_adjoint_cuda(g(x[0]), h, L))
    for i in range(2):
        rl, rh = w.mrdwt(x[0][i], h, L)
        assert relmax(yl[i].cpu().numpy(), rl) < 1e-5
        assert relmax(yh[i].cpu().numpy(), rh) < 1e-5
        assert relmax(back[i], w.mirdwt(x[0][i], y[i], h, L)) < 1e-5
        v, vh = x[1][i], rng.standard_normal((m, 3 * n * L))
        vl, vd = w.mrdwt(v, h, L)
        lhs, rhs = np.sum(xa[i] * v), np.sum(x[0][i] * vl) + np.sum(y[i] * vd)
        assert abs(lhs - rhs) < 1e-5 * np.linalg.norm(xa[i]) * np.linalg.norm(v)
        lhs, rhs = np.sum(al[i] * v) + np.sum(ah[i] * vh), np.sum(x[0][i] * w.mirdwt(v, vh, h, L))
        assert abs(lhs - rhs) < 1e-5 * np.hypot(np.linalg.norm(al[i]), np.linalg.norm(ah[i])) * np.hypot(
            np.linalg.norm(v), np.linalg.norm(vh))
