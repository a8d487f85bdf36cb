"""The 2^11-point-row FFT engine at the edges of its lengths: rows that just
fill a column count and the next one up, its shortest and longest rows and
the first on either side of them, both parities of n, both precisions, in
place and with strided rows, against scipy's DCT-I."""
import numpy as np
import pytest
import scipy.fft as sf

from tests.helpers import max_rel_err, rel_err
from tests.test_gpu_fft import gpu_dct1

pytestmark = pytest.mark.gpu

# column counts: one radix, two radices of every kind, the odd ones (a single
# self-paired row), the ends of the list
COUNTS = (2, 3, 5, 9, 15, 16, 18, 27, 40, 50, 64, 72, 81, 96, 100, 128, 144, 150, 180, 225, 240, 256)


@pytest.fixture(scope="module")
def env():
    import torch
    from minkasi_amd import device
    from minkasi_amd.lib import mkgpu
    return torch, device, mkgpu


def _rows(rng, rows, n):
    """A random walk plus white noise, as a detector mode."""
    return np.cumsum(rng.standard_normal((rows, n)), axis=1) * 0.006 + 0.1 * rng.standard_normal((rows, n))


@pytest.mark.parametrize("eb", [4, 8])
def test_filter_rows_at_length_edges(env, eb):
    torch, device, mkgpu = env
    from minkasi_amd.lib.plans import FiltPlan
    rng = np.random.default_rng(eb)
    dt = np.float32 if eb == 4 else np.float64
    # FP32: eps times the growth of a transform of 2^19 points on a red row
    # whose weights span the row's own power range; FP64 the same in its eps
    tol = 5e-6 if eb == 4 else 1e-12
    ns = [1365, 1366, 1367, 1368] + [2048 * q for q in COUNTS] + [2048 * q + 1 for q in COUNTS[::3]]
    for n in ns:
        x = _rows(rng, 2, n).astype(dt)
        w = 0.05 + np.abs(rng.standard_normal((2, n)))
        ref = sf.dct(sf.dct(x.astype(np.float64), type=1) * w, type=1)
        ref[:, [0, -1]] *= 0.5
        stride = n + 3
        buf = torch.full((2, stride), float("nan"), dtype=torch.float32 if eb == 4 else torch.float64,
                         device=device.device())
        buf[:, :n] = torch.from_numpy(x)
        wd = torch.from_numpy(sf.dct(w, type=1)).to(device.device())
        plan = FiltPlan([(2, n, 0, n, 0, n)], eb)
        plan.set_weights(wd)
        src = FiltPlan([(2, n, 0, stride, 0, stride)], eb)  # strided rows, borrowed spectra, in place
        src.borrow(0, plan, 0)
        src.set_halve(True)
        src.exec(buf, buf)
        out = buf.cpu().numpy()
        assert np.isnan(out[:, n:]).all(), n  # nothing written between the rows
        e, em = rel_err(out[:, :n], ref), max_rel_err(out[:, :n], ref)
        assert e < tol and em < 4 * tol, (n, e, em)
        plan.close()
        src.close()


def test_dct1_f64_at_length_edges(env):
    rng = np.random.default_rng(3)
    for q in COUNTS[::2]:
        for n in (1024 * q, 1024 * q + 1):  # 2(n-1)+1 points just fit 2^11 q, or need the next count
            x = rng.standard_normal((2, n))
            y, ref = gpu_dct1(env, x, np.float64), sf.dct(x, type=1)
            assert rel_err(y, ref) < 1e-13 and max_rel_err(y, ref) < 1e-12, n


def test_filter_rows_spread_a_nonfinite_sample_over_its_row_only(env):
    torch, device, mkgpu = env
    from minkasi_amd.lib.plans import FiltPlan
    n = 5000
    rng = np.random.default_rng(1)
    x = rng.standard_normal((3, n)).astype(np.float32)
    x[1, 0] = np.inf
    plan = FiltPlan([(3, n, 0, n, 0, n)], 4)
    plan.set_weights(torch.from_numpy(sf.dct(np.ones((3, n)), type=1)).to(device.device()))
    out = torch.empty(3, n, dtype=torch.float32, device=device.device())
    plan.exec(torch.from_numpy(x).to(device.device()), out)
    ok = torch.isfinite(out).all(dim=1).cpu().tolist()
    assert ok[0] and ok[2] and not ok[1]
