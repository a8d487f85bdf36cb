"""GPU parity of the learned-preconditioner kernels (conv3x3, adjoint weights,
wgrad, loss, Adam) and of the full forward/backward, through the C ABI,
against the FP64 oracle (oracle/learned.py).  FP32 on the GPU: tolerances are
stated per test."""
import numpy as np
import pytest

from oracle import learned as OL

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    import torch
    from minkasi_amd import device
    from minkasi_amd.lib import mkgpu
    return torch, device, mkgpu


def _t(env, a):
    torch, device, _ = env
    return device.to_device(np.ascontiguousarray(a, dtype=np.float32))


def rel(a, b):
    return float(np.linalg.norm(np.ravel(a) - np.ravel(b)) / max(np.linalg.norm(np.ravel(b)), 1e-300))


@pytest.mark.parametrize("cin,cout", [(1, 16), (16, 16), (16, 1), (1, 1)])
@pytest.mark.parametrize("dil", [1, 3, 27])
def test_conv3x3(env, cin, cout, dil):
    torch, device, mkgpu = env
    rng = np.random.default_rng(cin * 100 + cout + dil)
    B, H, W = 2, 37, 70
    x = rng.standard_normal((B, cin, H, W)).astype(np.float32)
    w = rng.standard_normal((cout, cin, 9)).astype(np.float32)
    ref = OL.conv3x3(x.astype(np.float64), w.astype(np.float64), dil)
    xt, wt = _t(env, x), _t(env, w)
    y = torch.full((B, cout, H, W), 7.0, dtype=torch.float32, device=xt.device)
    print("conv3x3", cin, cout, dil, flush=True)
    mkgpu.check("mk_conv3x3_f32", xt.data_ptr(), B, cin, H, W, wt.data_ptr(), cout, dil, y.data_ptr(), 0,
                device.stream_ptr())
    got = y.cpu().numpy()
    assert rel(got, ref) < 2e-6
    mkgpu.check("mk_conv3x3_f32", xt.data_ptr(), B, cin, H, W, wt.data_ptr(), cout, dil, y.data_ptr(), 1,
                device.stream_ptr())
    assert rel(y.cpu().numpy(), 2 * ref) < 2e-6


def test_conv3x3_adjoint_weights(env):
    torch, device, mkgpu = env
    rng = np.random.default_rng(1)
    w = rng.standard_normal((16, 1, 9)).astype(np.float32)
    wt = torch.empty(16 * 9, dtype=torch.float32, device=device.device())
    w_d = _t(env, w)
    mkgpu.check("mk_conv3x3_adjoint_weights", w_d.data_ptr(), 16, 1, wt.data_ptr(), device.stream_ptr())
    assert np.array_equal(wt.cpu().numpy().reshape(1, 16, 9), OL.adjoint_weights(w))


def test_conv3x3_rejects_bad_channels(env):
    torch, device, mkgpu = env
    x = torch.zeros(64, dtype=torch.float32, device=device.device())
    with pytest.raises(mkgpu.MkError):
        mkgpu.check("mk_conv3x3_f32", x.data_ptr(), 1, 3, 4, 4, x.data_ptr(), 16, 1, x.data_ptr() + 4, 0,
                    device.stream_ptr())


@pytest.mark.parametrize("co,ci", [(16, 16), (16, 1)])
@pytest.mark.parametrize("dil", [1, 9])
def test_wgrad(env, co, ci, dil):
    torch, device, mkgpu = env
    rng = np.random.default_rng(co + ci + dil)
    B, H, W = 3, 45, 52
    a = rng.standard_normal((B, co, H, W)).astype(np.float32)
    x = rng.standard_normal((B, ci, H, W)).astype(np.float32)
    ref = OL.wgrad(a.astype(np.float64), x.astype(np.float64), dil)
    nb = int(mkgpu.lib.mk_conv3x3_wgrad_workspace_bytes(B, co, ci, H, W, dil))
    work = torch.empty(nb // 4 + 1, dtype=torch.float32, device=device.device())
    g = torch.zeros(co * ci * 9, dtype=torch.float32, device=device.device())
    print("wgrad", co, ci, dil, flush=True)
    at, xt = _t(env, a), _t(env, x)  # keep both alive until the kernels have run
    mkgpu.check("mk_conv3x3_wgrad_f32", at.data_ptr(), co, xt.data_ptr(), ci, B, H, W, dil,
                g.data_ptr(), 0, work.data_ptr(), work.numel() * 4, device.stream_ptr())
    assert rel(g.cpu().numpy(), ref) < 1e-5
    mkgpu.check("mk_conv3x3_wgrad_f32", at.data_ptr(), co, xt.data_ptr(), ci, B, H, W, dil,
                g.data_ptr(), 1, work.data_ptr(), work.numel() * 4, device.stream_ptr())
    assert rel(g.cpu().numpy(), 2 * ref) < 1e-5


def _net_and_data(arch, spec, B, H, W, seed=0):
    from minkasi_amd.learned.precon import init_params, unpack
    rng = np.random.default_rng(seed)
    p = init_params(arch, spec, seed=seed, log_alpha=-0.3)
    ws, la = unpack(p, arch, len(spec))
    shp = (B, 1, H, W)
    r = rng.standard_normal(shp).astype(np.float32)
    e = rng.standard_normal(shp).astype(np.float32)
    s = rng.uniform(0.2, 1.5, shp).astype(np.float32)
    s[:, :, :3, :5] = 0.0
    m = (rng.uniform(size=shp) > 0.3).astype(np.float32)
    ws64 = [w.astype(np.float64) for w in ws]
    cls = {"chain": OL.Net, "levels": OL.LevelsNet, "tent": OL.TentLevelsNet}[arch]
    net = cls(ws64, spec, la)
    return p, net, r, e, s, m


ARCHS = [("chain", (1, 1, 1, 1)), ("chain", (1, 3, 9, 27)), ("levels", (1, 4, 16, 64)), ("levels", (1, 3, 6)),
         ("tent", (1, 4, 16, 64)), ("tent", (1, 3, 6))]


@pytest.mark.parametrize("arch,spec", ARCHS)
def test_forward_backward_vs_oracle(env, arch, spec):
    torch, device, mkgpu = env
    from minkasi_amd.learned.train import Trainer
    B, H, W = 2, 41, 66
    p, net, r, e, s, m = _net_and_data(arch, spec, B, H, W)
    loss, grads, dla = net.loss_and_grad(*(a.astype(np.float64) for a in (r, e, s, m)))
    tr = Trainer(p, arch, spec, B, H, W)
    print("forward_backward", arch, spec, flush=True)
    dev_in = [_t(env, a) for a in (r, e, s, m)]
    tr.forward_backward(*dev_in)
    torch.cuda.synchronize()
    assert abs(tr.loss() - loss) < 1e-5 * loss
    g = tr.grad.cpu().numpy()
    ref = np.concatenate([gr.ravel() for gr in grads])
    assert rel(g[:-1], ref) < 1e-4
    for (off, co, ci), gr in zip(tr.net.lay, grads):  # every layer on its own
        assert rel(g[off:off + co * ci * 9], gr.ravel()) < 2e-4
    alpha = np.exp(net.log_alpha)
    assert abs(alpha * tr.dalpha() - dla) < 1e-4 * abs(dla)


@pytest.mark.parametrize("arch,spec", [("chain", (1, 3, 9, 27)), ("levels", (1, 4, 16, 64)), ("tent", (1, 8, 32))])
def test_precon_apply_vs_oracle_and_symmetric(env, arch, spec):
    torch, device, mkgpu = env
    from minkasi_amd.learned.precon import LearnedPrecon
    H, W = 96, 130
    p, net, r, _, s, _ = _net_and_data(arch, spec, 1, H, W, seed=3)
    s00 = s[0, 0].astype(np.float64)
    hits = np.where(s00 > 0, 1.0 / np.where(s00 > 0, s00, 1.0) ** 2, 0.0).astype(np.float32)
    lp = LearnedPrecon(_t(env, hits), p, arch, spec)
    s_used = lp.s.cpu().numpy().astype(np.float64)
    rt = _t(env, r[0, 0])
    z = torch.empty_like(rt)
    lp.apply_to(rt, z)
    ref = net.apply(r[0, 0].astype(np.float64), s_used)
    assert rel(z.cpu().numpy(), ref) < 1e-5
    rng = np.random.default_rng(9)
    x = rng.standard_normal((H, W)).astype(np.float32)
    y = rng.standard_normal((H, W)).astype(np.float32)
    mx, my = torch.empty_like(rt), torch.empty_like(rt)
    xd, yd = _t(env, x), _t(env, y)
    lp.apply_to(xd, mx)
    lp.apply_to(yd, my)
    a = float(np.dot(x.ravel().astype(np.float64), my.cpu().numpy().ravel()))
    b = float(np.dot(mx.cpu().numpy().ravel().astype(np.float64), y.ravel()))
    xmx = float(np.dot(x.ravel().astype(np.float64), mx.cpu().numpy().ravel()))
    ymy = float(np.dot(y.ravel().astype(np.float64), my.cpu().numpy().ravel()))
    assert abs(a - b) < 1e-5 * np.sqrt(abs(xmx * ymy))
    assert xmx > 0


@pytest.mark.parametrize("kind,f", [("box", 4), ("tent", 4), ("tent", 3), ("tent", 8)])
def test_restrict_prolong(env, kind, f):
    torch, device, mkgpu = env
    rng = np.random.default_rng(13 + f)
    B, H, W = 2, 37, 45
    x = rng.standard_normal((B, 1, H, W)).astype(np.float32)
    y = rng.standard_normal((B, 1, -(-H // f), -(-W // f))).astype(np.float32)
    xd, yd = _t(env, x), _t(env, y)
    ry = torch.empty_like(yd)
    R, Pr = (OL.restrict, OL.prolong) if kind == "box" else (OL.restrict_tent, OL.prolong_tent)
    mkgpu.check("mk_restrict_%s_f32" % kind, xd.data_ptr(), B, H, W, f, ry.data_ptr(), device.stream_ptr())
    assert rel(ry.cpu().numpy(), R(x, f)) < 1e-6
    px = torch.full_like(xd, 2.0)
    mkgpu.check("mk_prolong_%s_f32" % kind, yd.data_ptr(), B, H, W, f, px.data_ptr(), 1, device.stream_ptr())
    assert rel(px.cpu().numpy(), 2.0 + Pr(y, f, H, W)) < 1e-6


def test_adam_matches_numpy(env):
    torch, device, mkgpu = env
    rng = np.random.default_rng(4)
    n = 1000
    p = rng.standard_normal(n).astype(np.float32)
    g = rng.standard_normal(n).astype(np.float32)
    dal = np.array([0.7, 0.0])
    pt, gt = _t(env, p), _t(env, g)
    mt = torch.zeros_like(pt)
    vt = torch.zeros_like(pt)
    dt = device.to_device(dal)
    pr, m, v = p.astype(np.float64), np.zeros(n), np.zeros(n)
    lr, b1, b2, eps = 1e-2, 0.9, 0.999, 1e-8
    for step in (1, 2, 3):
        mkgpu.check("mk_adam_f32", pt.data_ptr(), gt.data_ptr(), mt.data_ptr(), vt.data_ptr(), n, dt.data_ptr(),
                    lr, b1, b2, eps, step, 0.5, device.stream_ptr())
        gg = 0.5 * g.astype(np.float64)
        gg[-1] = 0.5 * np.exp(pr[-1]) * dal[0]
        m = b1 * m + (1 - b1) * gg
        v = b2 * v + (1 - b2) * gg * gg
        pr = pr - lr * (m / (1 - b1 ** step)) / (np.sqrt(v / (1 - b2 ** step)) + eps)
    assert np.max(np.abs(pt.cpu().numpy() - pr)) < 1e-5


@pytest.mark.parametrize("arch,spec", [("chain", (1, 2, 1, 3)), ("levels", (1, 2, 4))])
def test_energy_forward_backward_vs_oracle(env, arch, spec):
    torch, device, mkgpu = env
    from minkasi_amd.learned.train import Trainer
    H, W = 14, 11
    n = H * W
    p, net, _, _, s, _ = _net_and_data(arch, spec, 1, H, W, seed=5)
    rng = np.random.default_rng(8)
    Q = rng.standard_normal((n, n))
    A = Q @ Q.T / n + 0.05 * np.eye(n)
    e = rng.standard_normal((H, W))
    r = (A @ e.ravel()).reshape(H, W)
    s2 = s[0, 0].astype(np.float64)
    loss, grads, dla = net.energy_loss_and_grad(r, e, s2, A)
    At = device.to_device(A.astype(np.float32))

    def apply_A(z, out):  # dense test operator
        out.copy_((At @ z.reshape(-1)).reshape(H, W))

    tr = Trainer(p, arch, spec, 1, H, W)
    ins = [_t(env, a) for a in (r, e, s2)]
    print("energy_forward_backward", arch, spec, flush=True)
    tr.energy_forward_backward(ins[0], ins[1], ins[2], apply_A)
    torch.cuda.synchronize()
    assert abs(tr.loss() - loss) < 1e-4 * loss
    g = tr.grad.cpu().numpy()
    ref = np.concatenate([gr.ravel() for gr in grads])
    assert rel(g[:-1], ref) < 1e-4
    assert abs(np.exp(net.log_alpha) * tr.dalpha() - dla) < 1e-4 * abs(dla)


@pytest.mark.parametrize("fname,arch_want,max_ratio", [("weights_c4.npz", "tent", 0.75),
                                                     ("weights_c4_chain.npz", "chain", 0.9)])
def test_shipped_weights_gain_over_jacobi(env, fname, arch_want, max_ratio):
    """What the trained networks gain over the method without them: the
    shipped weights (minkasi_amd/learned/weights_c4.npz, the multilevel net,
    and weights_c4_chain.npz, the 4-layer chain), on a 16-TOD problem of the
    benchmark's distribution with seeds used neither in training nor in
    calibration, reach ||r||/||b|| < 1e-6 in fewer PCG iterations than the
    hits-count Jacobi preconditioner alone, to the same solution.  The
    preconditioner they define is symmetric and positive on hit pixels."""
    torch, device, mkgpu = env
    import os
    from minkasi_amd.learned.precon import LearnedPrecon, load
    from minkasi_amd.synth import tod_shapes
    from minkasi_amd.workloads import build_problem, map_distance, solve_to_tol
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "minkasi_amd", "learned",
                        fname)
    params, arch, spec, meta = load(path)
    assert arch == arch_want
    P = build_problem(4, shapes=tod_shapes(4, 16, seed=777), seed_base=5_000_000)
    lp = LearnedPrecon(P.hits, params, arch, spec)
    hit = P.hits.map > 0
    g = torch.Generator(device=P.hits.map.device).manual_seed(3)
    x = torch.randn(P.hits.map.shape, device=P.hits.map.device, generator=g) * hit
    y = torch.randn(P.hits.map.shape, device=P.hits.map.device, generator=g) * hit
    mx, my = torch.empty_like(x), torch.empty_like(y)
    lp.apply_to(x, mx)
    lp.apply_to(y, my)
    a, b = float((y.double() * mx.double()).sum()), float((x.double() * my.double()).sum())
    assert abs(a - b) < 1e-4 * abs(a) and float((x.double() * mx.double()).sum()) > 0
    jac = solve_to_tol(P, None, 1e-6, 400)
    lrn = solve_to_tol(P, lp, 1e-6, 400)
    print("16-TOD held-out problem: Jacobi %d its %.2f s, learned %d its %.2f s" % (
        jac["iters"], jac["seconds"], lrn["iters"], lrn["seconds"]))
    assert jac["reached"] and lrn["reached"]
    assert lrn["iters"] <= max_ratio * jac["iters"], (lrn["iters"], jac["iters"])
    assert lrn["true_rel_res"] < 3e-6
    assert map_distance(P, lrn["x"], jac["x"]) < 1e-3


# Edges of the composed-stencil path: images thinner than the stencil, tiles
# of 64 x 8 and (from 512 of them) 64 x 32 pixels with remainders, odd and unit
# steps, a coarse level narrower than its support, and coarse levels inside and
# outside the one-workgroup tail.  1e-5: a few hundred FP32 roundings of 6e-8
# at worst.
@pytest.mark.parametrize("arch,spec,B,H,W", [
    ("tent", (1,), 1, 1, 1), ("levels", (1, 2), 3, 1, 9), ("tent", (1, 2, 6), 1, 2, 3), ("tent", (1, 1, 4), 1, 7, 64),
    ("levels", (1, 3, 6, 12), 2, 33, 65), ("tent", (1, 4, 16, 64, 256), 1, 129, 257), ("tent", (1, 64), 1, 130, 200),
    ("levels", (1, 64, 128), 1, 65, 1000), ("tent", (1, 3), 90, 65, 70), ("levels", (1, 4, 16), 1, 1031, 1025),
    ("tent", (1, 5, 10, 20), 1, 300, 31)])
def test_levels_precon_edges(env, arch, spec, B, H, W):
    torch, device, mkgpu = env
    from minkasi_amd.learned.nets import make_net
    p, net, r, _, s, _ = _net_and_data(arch, spec, B, H, W, seed=H + W)
    s = s + np.float32(0.1)  # no pixel is masked: the smallest images are all corner
    gnet = make_net(arch, spec, p, B, H, W)
    gnet.refresh_adjoint()
    rt, st = _t(env, r), _t(env, s)
    z = torch.full_like(rt, 3.0)
    print("levels_precon", arch, spec, B, H, W, flush=True)
    gnet.precondition(rt, st, z)
    ref = net.apply(r.astype(np.float64), s.astype(np.float64))
    assert np.linalg.norm(z.cpu().numpy() - ref) <= 1e-5 * np.linalg.norm(ref)


def test_levels_precon_in_place(env):
    torch, device, mkgpu = env
    from minkasi_amd.learned.precon import LearnedPrecon
    p, net, r, _, s, _ = _net_and_data("tent", (1, 4), 1, 41, 66)
    lp = LearnedPrecon(_t(env, s[0, 0]), p, "tent", (1, 4))
    rt = _t(env, r[0, 0])
    z = torch.empty_like(rt)
    lp.apply_to(rt, z)
    lp.apply_to(rt, rt)
    assert torch.equal(rt, z)


@pytest.mark.parametrize("arch,spec", [("levels", (1, 2)), ("tent", (1, 4, 16))])
def test_levels_forward_outside_training(env, arch, spec):
    """The layered K^T K u of a network built without training buffers is the
    training network's, and leaves precondition() as it was."""
    torch, device, mkgpu = env
    from minkasi_amd.learned.nets import make_net
    p, _, r, _, s, _ = _net_and_data(arch, spec, 2, 37, 50)
    u, out = _t(env, r * s), []
    for train in (True, False):
        net = make_net(arch, spec, p, 2, 37, 50, train)
        for scale in (1.0, -0.5):  # new weights reach the adjoint layers too
            net.params.mul_(scale)
            net.refresh_adjoint()
            g = torch.full_like(u, 3.0)
            net.forward(u, g)
            out.append(g)
    assert torch.equal(out[0], out[2]) and torch.equal(out[1], out[3])
    assert not torch.equal(out[0], out[1])
    z = [torch.empty_like(u) for _ in range(2)]
    for zi in z:
        net.precondition(_t(env, r), _t(env, s), zi)
        net.forward(u, g)
    assert torch.equal(z[0], z[1])


def test_levels_forward_replayed_with_new_weights(env):
    """A captured forward() outside training reads the weights of the last
    refresh_adjoint() at every replay."""
    torch, device, mkgpu = env
    from minkasi_amd.learned.nets import make_net
    p, _, r, _, s, _ = _net_and_data("tent", (1, 4), 1, 37, 50)
    net = make_net("tent", (1, 4), p, 1, 37, 50)
    net.refresh_adjoint()
    u = _t(env, r * s)
    g, want = torch.empty_like(u), torch.empty_like(u)
    net.forward(u, g)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        net.forward(u, g)
    for scale in (1.0, -0.5, 3.0):
        net.params.mul_(scale)
        net.refresh_adjoint()
        graph.replay()
        torch.cuda.synchronize()
        got = g.clone()
        net.forward(u, want)
        assert torch.equal(got, want)
