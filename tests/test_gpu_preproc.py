"""Device TOD preprocessing (fit_cm_plus_poly, downsample_tod) against the
FP64 oracle (oracle/preproc.py) and numpy."""
import numpy as np
import pytest

from oracle import preproc as opre
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from minkasi_amd import device
    from minkasi_amd.lib import mkgpu
    return torch, device, mkgpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_median_cols_equals_numpy(env, dtype):
    torch, device, mkgpu = env
    rng = np.random.default_rng(0)
    sfx = "f64" if dtype == np.float64 else "f32"
    for nrow in (1, 2, 3, 63, 64, 65, 100, 128, 511, 512, 513, 1000, 1024):
        for ncol in (1, 5, 777):
            ld = ncol + 3
            a = rng.standard_normal((nrow, ld)).astype(dtype)
            a[:, ::7] = np.round(a[:, ::7])  # ties
            at = device.to_device(a)
            out = torch.empty(ncol, dtype=at.dtype, device=at.device)
            mkgpu.check("mk_median_cols_" + sfx, at.data_ptr(), nrow, ncol, ld, out.data_ptr(), device.stream_ptr())
            ref = np.median(a[:, :ncol], axis=0)
            assert np.array_equal(out.cpu().numpy(), ref.astype(dtype)), (nrow, ncol)


def _data(ndet, n, seed):
    rng = np.random.default_rng(seed)
    cm = np.cumsum(rng.standard_normal(n)) * 0.05
    x = np.linspace(-1, 1, n)
    drift = rng.standard_normal((ndet, 3)) @ np.stack([np.ones(n), x, x ** 2])
    return (1 + 0.05 * rng.standard_normal((ndet, 1))) * cm + drift + 0.1 * rng.standard_normal((ndet, n))


@pytest.mark.parametrize("ndet,n,ord,cm_ord,niter", [(64, 20001, 2, 1, 1), (215, 9000, 3, 2, 2), (7, 1001, 0, 1, 1),
                                                      (512, 40000, 2, 1, 1)])
def test_fit_cm_plus_poly_matches_oracle(env, ndet, n, ord, cm_ord, niter):
    torch, device, mkgpu = env
    from minkasi_amd.tods.processing import fit_cm_plus_poly
    dat = _data(ndet, n, ndet + n)
    dd_r, p2_r, cm_r = opre.fit_cm_plus_poly(dat, ord, cm_ord, niter, full_out=True)
    dd, p2, cm = fit_cm_plus_poly(device.to_device(dat), ord, cm_ord, niter, full_out=True)
    assert rel_err(dd.cpu().numpy(), dd_r) < 1e-10
    assert rel_err(p2.cpu().numpy(), p2_r) < 1e-10
    assert np.array_equal(cm.cpu().numpy(), cm_r) or niter > 1
    if niter == 1:
        d32 = fit_cm_plus_poly(device.to_device(dat.astype(np.float32)), ord, cm_ord, niter)
        ref32 = opre.fit_cm_plus_poly(dat.astype(np.float32).astype(np.float64), ord, cm_ord, niter)
        assert d32.dtype == torch.float32
        assert rel_err(d32.cpu().numpy(), ref32) < 1e-5
    host = fit_cm_plus_poly(dat, ord, cm_ord, niter)  # numpy in, FP64 numpy out
    assert isinstance(host, np.ndarray) and host.dtype == np.float64
    assert rel_err(host, dd_r) < 1e-10


def test_fit_cm_plus_poly_exact_when_median_is_known(env):
    torch, device, mkgpu = env
    from minkasi_amd.tods.processing import fit_cm_plus_poly
    rng = np.random.default_rng(4)
    n = 5000
    m = np.cumsum(rng.standard_normal(n)) * 0.1
    x = np.linspace(-1, 1, n)
    dat = np.stack([m, m + 2 + 0.5 * x + 0.3 * x ** 2, m + 3 - x, m - 1.5 - 0.2 * x ** 2, m - 2.5 - x ** 2])
    dd, p2, cm = fit_cm_plus_poly(device.to_device(dat), 2, 1, full_out=True)
    assert np.array_equal(cm.cpu().numpy(), m)
    assert np.max(np.abs(dd.cpu().numpy() - m)) < 1e-10
    assert np.max(np.abs(p2.cpu().numpy() - m)) < 1e-10


def test_downsample_tod_matches_oracle(env):
    torch, device, mkgpu = env
    from minkasi_amd.tods.processing import downsample_tod
    rng = np.random.default_rng(5)
    ndet, n = 6, 30001
    dat = rng.standard_normal((ndet, n))
    ra = np.linspace(0, 1, n)
    info = {"dat_calib": device.to_device(dat), "ra_b": ra.copy(), "dra": rng.standard_normal(ndet), "dt": 0.01}
    downsample_tod(info, 10)
    nn = n // 10
    assert abs(info["dt"] - 0.1) < 1e-15
    assert tuple(info["dat_calib"].shape) == (ndet, nn)
    assert rel_err(info["dat_calib"].cpu().numpy(), opre.downsample_array(dat, 10)) < 1e-12
    assert info["ra_b"].shape == (nn,) and rel_err(info["ra_b"], opre.downsample_array(ra, 10)) < 1e-12
    assert info["dra"].shape == (ndet,)
    d32 = {"dat_calib": device.to_device(dat.astype(np.float32)), "dt": 1.0}
    downsample_tod(d32, 4)
    assert rel_err(d32["dat_calib"].cpu().numpy(), opre.downsample_array(dat.astype(np.float32), 4)) < 2e-6


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nrow", [1, 2, 5, 64, 130, 700, 1024])
def test_median_cols_extreme_values(env, dtype, nrow):
    """Infinities, equal values, zeros of both signs, subnormals, and a range
    that spans every exponent: the order statistics are exact."""
    torch, device, mkgpu = env
    rng = np.random.default_rng(nrow)
    tiny = np.finfo(dtype).tiny
    a = rng.standard_normal((nrow, 33)).astype(dtype)
    a[:, 0] = 3.25
    a[:, 1] = np.inf
    a[:, 2] = -np.inf
    a[: nrow // 3, 3] = np.inf
    a[: nrow // 3, 4] = -np.inf
    a[:, 5] = np.where(np.arange(nrow) % 2, 0.0, -0.0)
    a[:, 6] = rng.integers(-3, 4, nrow) * (tiny / 4)
    a[:, 7] = rng.integers(0, 2, nrow)
    a[:, 8] = np.exp(rng.uniform(-80, 80, nrow)) * rng.choice([-1, 1], nrow)
    a[:, 9] = -np.abs(a[:, 9])
    at = device.to_device(a)
    out = torch.empty(33, dtype=at.dtype, device=at.device)
    print("median", dtype.__name__, nrow, flush=True)
    mkgpu.check("mk_median_cols_" + ("f64" if dtype == np.float64 else "f32"), at.data_ptr(), nrow, 33, 33,
                out.data_ptr(), device.stream_ptr())
    srt = np.sort(a, axis=0)
    ref = srt[nrow // 2] if nrow % 2 else (srt[nrow // 2 - 1] + srt[nrow // 2]) / dtype(2)
    got = out.cpu().numpy()
    assert np.array_equal(got[[0, 1, 2, 3, 4, 5, 7, 8, 9]], ref[[0, 1, 2, 3, 4, 5, 7, 8, 9]])
    assert abs(got[6] - ref[6]) <= tiny / 8  # the halved sum of an odd subnormal sum rounds to either side
    assert np.array_equal(got[10:], ref[10:])


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nrow", [1, 2, 9, 64, 65, 215, 1024])
def test_median_cols_nan(env, dtype, nrow):
    """A column with a NaN of either sign and any payload has a NaN median, as
    np.median gives; its neighbours do not."""
    torch, device, mkgpu = env
    rng = np.random.default_rng(nrow)
    a = rng.standard_normal((nrow, 12)).astype(dtype)
    u = a.view(np.uint32 if dtype == np.float32 else np.uint64)
    top = np.finfo(dtype).bits - 1
    inf = int(np.array(np.inf, dtype=dtype).view(u.dtype))
    for c, bits in ((1, inf + 1), (3, inf + 1 + (1 << top)), (5, (1 << top) - 1), (7, (2 << top) - 1)):
        u[rng.integers(nrow), c] = bits
    a[:, 9] = np.nan
    a[nrow // 2:, 10] = np.inf
    a[0, 10] = np.nan
    at = device.to_device(a)
    out = torch.empty(12, dtype=at.dtype, device=at.device)
    print("median nan", dtype.__name__, nrow, flush=True)
    mkgpu.check("mk_median_cols_" + ("f64" if dtype == np.float64 else "f32"), at.data_ptr(), nrow, 12, 12,
                out.data_ptr(), device.stream_ptr())
    got = out.cpu().numpy()
    assert np.array_equal(got, np.median(a, axis=0), equal_nan=True)
    assert np.array_equal(np.isnan(got), np.isin(np.arange(12), [1, 3, 5, 7, 9, 10]))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nrow", [3, 63, 64, 65])
@pytest.mark.parametrize("ncol", [1, 4099, 8191, 8193, 16385, 32769])
def test_median_cols_column_groups(env, dtype, nrow, ncol):
    """4 to 32 columns per workgroup with remainders, on both sides of the 64
    rows that are sorted and not bisected."""
    torch, device, mkgpu = env
    a = np.random.default_rng(nrow + ncol).integers(-40, 40, (nrow, ncol + 3)).astype(dtype) / 8  # ties
    at = device.to_device(a)
    out = torch.full((ncol + 1,), 9.0, dtype=at.dtype, device=at.device)
    print("median groups", dtype.__name__, nrow, ncol, flush=True)
    mkgpu.check("mk_median_cols_" + ("f64" if dtype == np.float64 else "f32"), at.data_ptr(), nrow, ncol, ncol + 3,
                out.data_ptr(), device.stream_ptr())
    got = out.cpu().numpy()
    assert got[ncol] == 9.0
    assert np.array_equal(got[:ncol], np.median(a[:, :ncol], axis=0))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nrow,n,ncol", [(1, 1, 1), (7, 255, 2), (8, 256, 3), (9, 257, 5), (17, 4096, 6), (5, 4097, 7),
                                         (16, 9001, 8), (3, 300, 11)])
def test_design_dots_and_apply_edges(env, dtype, nrow, n, ncol):
    """Row groups of 8 and sample chunks of 256 and 4096 with remainders.
    FP64 sums: n eps of the sum of magnitudes (1e-12); the subtraction rounds
    once more in the data type."""
    torch, device, mkgpu = env
    sfx = "f64" if dtype == np.float64 else "f32"
    rng = np.random.default_rng(nrow + n + ncol)
    X, ld = rng.standard_normal((n, ncol)), n + 5
    y = rng.standard_normal((nrow, ld)).astype(dtype)
    Xt, yt = device.to_device(X), device.to_device(y)
    f64 = dict(dtype=torch.float64, device=yt.device)
    sp = device.stream_ptr()
    print("design", sfx, nrow, n, ncol, flush=True)
    if ncol <= 8:
        nb = int(mkgpu.lib.mk_design_dots_workspace_bytes(n, ncol, nrow))
        work, D = torch.empty(nb // 8, **f64), torch.empty((ncol, nrow), **f64)
        mkgpu.check("mk_design_dots_" + sfx, Xt.data_ptr(), n, ncol, yt.data_ptr(), nrow, ld, D.data_ptr(),
                    work.data_ptr(), nb // 8 * 8, sp)
        ref = X.T @ y[:, :n].astype(np.float64).T
        assert np.all(np.abs(D.cpu().numpy() - ref) <= 1e-12 * (np.abs(X.T) @ np.abs(y[:, :n].astype(np.float64).T)))
    c0 = min(1, ncol - 1)
    coef = rng.standard_normal((ncol - c0, nrow))
    ct = device.to_device(coef)
    p = (X[:, c0:] @ coef).T
    eps = np.finfo(dtype).eps
    for base in (True, False):
        out = torch.full((nrow, n + 2), 9.0, dtype=yt.dtype, device=yt.device)
        mkgpu.check("mk_design_apply_" + sfx, yt.data_ptr() if base else 0, nrow, n, ld, Xt.data_ptr(), ncol, c0,
                    ncol - c0, ct.data_ptr(), out.data_ptr(), n + 2, sp)
        ref = y[:, :n].astype(np.float64) - p if base else p
        got = out.cpu().numpy()
        assert np.all(got[:, n:] == 9.0)
        assert np.all(np.abs(got[:, :n] - ref) <= eps * (np.abs(ref) + 20 * np.finfo(np.float64).eps / eps * 100))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nrow,n,ncol", [(1, 511, 6), (6, 33300, 6), (64, 513, 8), (64, 65537, 3), (130, 40001, 2),
                                         (520, 33000, 1)])
def test_design_dots_chunks(env, dtype, nrow, n, ncol):
    """Chunks of 512, 1024, 2048 and 4096 samples and more of them than a wave
    has lanes.  A sum passes at most 16 + 6 + 4 + 8 + 6 additions on its way
    and a product rounds once: 41 eps of the sum of magnitudes."""
    torch, device, mkgpu = env
    rng = np.random.default_rng(nrow + n + ncol)
    X, y = rng.standard_normal((n, ncol)), rng.standard_normal((nrow, n)).astype(dtype)
    Xt, yt = device.to_device(X), device.to_device(y)
    nb = int(mkgpu.lib.mk_design_dots_workspace_bytes(n, ncol, nrow))
    work = torch.empty(nb // 8, dtype=torch.float64, device=yt.device)
    D = torch.empty((ncol, nrow), dtype=torch.float64, device=yt.device)
    print("design chunks", dtype.__name__, nrow, n, ncol, flush=True)
    for _ in range(2):  # the sums repeat bitwise
        prev = D.clone()
        mkgpu.check("mk_design_dots_" + ("f64" if dtype == np.float64 else "f32"), Xt.data_ptr(), n, ncol,
                    yt.data_ptr(), nrow, n, D.data_ptr(), work.data_ptr(), nb, device.stream_ptr())
    assert torch.equal(prev, D)
    y64 = y.astype(np.longdouble)
    ref, mag = X.T.astype(np.longdouble) @ y64.T, np.abs(X.T) @ np.abs(y64.T)
    assert np.all(np.abs(D.cpu().numpy() - ref) <= 41 * np.finfo(np.float64).eps * mag)
