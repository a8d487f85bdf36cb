"""FP64 products and smoothing of the noise-model setup at the edges of their
tiles, against numpy in FP64.  A sum of K rounded products is within K eps of
the sum of magnitudes; 1e-13 of it covers the longest one here."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from minkasi_amd import device
    from minkasi_amd.lib import mkgpu
    return torch, device, mkgpu


def _close(got, ref, mag):
    assert np.all(np.abs(got - ref) <= 1e-13 * mag)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("M,K,N", [(1, 1, 1), (15, 3, 63), (16, 4, 64), (17, 5, 65), (32, 16, 130), (33, 17, 257),
                                   (64, 31, 255), (65, 64, 66), (129, 215, 301)])
def test_gemm_nn_edges(env, dtype, M, K, N):
    torch, device, mkgpu = env
    rng = np.random.default_rng(M + K + N)
    lda, ldb, ldc = K + 1, N + 3, N + 2
    A, B = rng.standard_normal((M, lda)), rng.standard_normal((K, ldb)).astype(dtype)
    A[:, K:], B[:, N:] = np.nan, np.nan  # nothing beyond the operands is used
    At, Bt = device.to_device(A), device.to_device(B)
    C = torch.full((M, ldc), 9.0, dtype=torch.float64, device=At.device)
    print("gemm", dtype.__name__, M, K, N, flush=True)
    mkgpu.check("mk_gemm_nn_f64", M, N, K, At.data_ptr(), lda, Bt.data_ptr(), int(dtype == np.float32), ldb,
                C.data_ptr(), ldc, device.stream_ptr())
    a, b, got = A[:, :K], B[:, :N].astype(np.float64), C.cpu().numpy()
    assert np.all(got[:, N:] == 9.0)
    _close(got[:, :N], a @ b, np.abs(a) @ np.abs(b))


@pytest.mark.parametrize("K", [1, 16, 17, 32, 33])
@pytest.mark.parametrize("N", [1, 2, 3, 31, 33, 62, 63, 66, 67, 97, 125])
def test_gemm_nn_column_groups(env, K, N):
    """Pairs (K up to 32) and fours of columns per lane, at every remainder."""
    torch, device, mkgpu = env
    M, ldc = 37, N + 1
    rng = np.random.default_rng(K + 100 * N)
    A = rng.standard_normal((M, K))
    At = device.to_device(A)
    print("gemm groups", K, N, flush=True)
    for dtype in (np.float32, np.float64):
        B = rng.standard_normal((K, N)).astype(dtype)
        Bt = device.to_device(B)
        C = torch.full((M, ldc), 9.0, dtype=torch.float64, device=At.device)
        mkgpu.check("mk_gemm_nn_f64", M, N, K, At.data_ptr(), K, Bt.data_ptr(), int(dtype == np.float32), N,
                    C.data_ptr(), ldc, device.stream_ptr())
        b, got = B.astype(np.float64), C.cpu().numpy()
        assert np.all(got[:, N:] == 9.0)
        _close(got[:, :N], A @ b, np.abs(A) @ np.abs(b))


@pytest.mark.parametrize("M,N,n", [(1, 1, 1), (16, 17, 15), (31, 33, 16), (64, 65, 1025), (65, 3, 2049), (130, 70, 5003)])
def test_cross_and_gram_edges(env, M, N, n):
    torch, device, mkgpu = env
    rng = np.random.default_rng(M + N + n)
    A, B = rng.standard_normal((M, n)), rng.standard_normal((N, n))
    At, Bt = device.to_device(A), device.to_device(B)
    f64 = dict(dtype=torch.float64, device=At.device)
    sp = device.stream_ptr()
    nb = int(mkgpu.lib.mk_cross_workspace_bytes(M, N, n))
    C, work = torch.empty((M, N), **f64), torch.empty(nb // 8, **f64)
    print("cross", M, N, n, flush=True)
    mkgpu.check("mk_cross_f64", M, N, n, At.data_ptr(), n, Bt.data_ptr(), n, C.data_ptr(), work.data_ptr(), nb, sp)
    _close(C.cpu().numpy(), A @ B.T, np.abs(A) @ np.abs(B).T)
    nb = int(mkgpu.lib.mk_gram_workspace_bytes(M, n))
    for dtype in (np.float32, np.float64):
        D = A.astype(dtype)
        Dt = device.to_device(D)
        G, work = torch.full((M, M), 5.0, **f64), torch.empty(nb // 8, **f64)
        mkgpu.check("mk_gram_f64", M, n, Dt.data_ptr(), int(dtype == np.float32), n, G.data_ptr(), work.data_ptr(),
                    nb, sp)
        d, got = D.astype(np.float64), G.cpu().numpy()
        _close(got, d @ d.T, np.abs(d) @ np.abs(d).T)
        assert np.array_equal(got, got.T)


@pytest.mark.parametrize("n,t_lo,t_hi", [(2, 0, 0), (2, 0, 1), (9, -7, 8), (100, -6, 7), (1023, -8, 7), (1024, -4, 4),
                                         (1025, -276, 276), (2500, -3, 20), (3000, -2998, 2999), (9000, -8192, 8192)])
def test_smooth_rows_edges(env, n, t_lo, t_hi):
    """The circular sum over the taps of the even extension, tap counts with
    every kind of remainder, up to the largest window."""
    torch, device, mkgpu = env
    rng = np.random.default_rng(n)
    x, g = rng.standard_normal((3, n)), rng.uniform(0.1, 1.0, max(t_hi, -t_lo) + 1)
    xt, gt = device.to_device(x), device.to_device(g)
    out = torch.empty_like(xt)
    print("smooth", n, t_lo, t_hi, flush=True)
    mkgpu.check("mk_smooth_rows_f64", xt.data_ptr(), out.data_ptr(), 0, 3, n, gt.data_ptr(), t_lo, t_hi, 0,
                device.stream_ptr())
    m, k = n - 1, np.arange(n)
    ref, mag = np.zeros((3, n)), np.zeros((3, n))
    for t in range(t_lo, t_hi + 1):
        i = np.abs(k - t)
        v = x[:, np.where(i > m, 2 * m - i, i)]
        ref += g[abs(t)] * v
        mag += g[abs(t)] * np.abs(v)
    assert np.all(np.abs(out.cpu().numpy() - ref) <= 1e-12 * mag)  # up to 16385 terms on both sides


def test_cross_and_gram_in_a_longer_calls_workspace(env):
    """511 chunks of 8192 samples are split into shorter ones, 512 are not: the
    shorter call still runs in the longer one's workspace."""
    torch, device, mkgpu = env
    n = 511 * 8192
    rng = np.random.default_rng(5)
    A, B = rng.standard_normal((1, n)), rng.standard_normal((2, n))
    At, Bt = device.to_device(A), device.to_device(B)
    f64 = dict(dtype=torch.float64, device=At.device)
    sp = device.stream_ptr()
    for got, size, call, ref, mag in (
            (torch.empty((1, 2), **f64), mkgpu.lib.mk_cross_workspace_bytes(1, 2, n + 8192),
             lambda C, w, nb: mkgpu.check("mk_cross_f64", 1, 2, n, At.data_ptr(), n, Bt.data_ptr(), n, C.data_ptr(),
                                          w.data_ptr(), nb, sp), A @ B.T, np.abs(A) @ np.abs(B).T),
            (torch.empty((2, 2), **f64), mkgpu.lib.mk_gram_workspace_bytes(2, n + 8192),
             lambda C, w, nb: mkgpu.check("mk_gram_f64", 2, n, Bt.data_ptr(), 0, n, C.data_ptr(), w.data_ptr(), nb,
                                          sp), B @ B.T, np.abs(B) @ np.abs(B).T)):
        work = torch.empty(int(size) // 8, **f64)
        call(got, work, int(size))
        _close(got.cpu().numpy(), ref, mag)
