"""Reprojection adjoint behind torch.autograd.Function: the GPU backward
kernels against central finite differences of the FP64 oracle residual
(h = 1e-4) and against the FP64 analytic Jacobians (g2o linearizeOplus)."""
import numpy as np
import pytest

import oracle
from kernel_check import device_events
from mcvslam_amd import BALinearizer, synth
from mcvslam_amd.autograd import apply_increments, reprojection

pytestmark = pytest.mark.gpu


def _problem():
    return synth.ba_problem(seed=34, n_kf=4, n_points=1500, target_obs=12000)


def _oracle_e(prob, dpose, dpoint):
    pts, frs = apply_increments(prob.points, prob.frames, dpose, dpoint)
    p = synth.BAProblem(**{k: np.copy(v) for k, v in prob.__dict__.items()})
    p.points, p.frames = pts, frs
    return oracle.ba_linearize(p)[0]


def test_adjoint_vs_fd_and_jacobians(gpu_ctx):
    import torch
    prob = _problem()
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P, M = len(prob.frames), len(prob.points), len(prob.obs_pt)
    dpose = torch.zeros((F, 6), dtype=torch.float64, device="cuda", requires_grad=True)
    dpoint = torch.zeros((P, 3), dtype=torch.float64, device="cuda", requires_grad=True)
    e = reprojection(dpose, dpoint, lin, (prob.points, prob.frames, prob.cams))
    rng = np.random.default_rng(0)
    G = rng.normal(size=(M, 2))
    (e * torch.from_numpy(G).float().cuda()).sum().backward()
    gpose = dpose.grad.cpu().numpy()
    gpoint = dpoint.grad.cpu().numpy()
    # FP64 analytic adjoint from the oracle's Jacobians
    _, _, _, Jp, Jx = oracle.ba_linearize(prob)
    want_pose = np.zeros((F, 6))
    want_point = np.zeros((P, 3))
    np.add.at(want_pose, prob.obs_frame, np.einsum("mij,mi->mj", Jp, G))
    np.add.at(want_point, prob.obs_pt, np.einsum("mij,mi->mj", Jx, G))
    for got, want in ((gpose, want_pose), (gpoint, want_point)):
        err = np.linalg.norm(got - want, axis=1) / np.maximum(np.linalg.norm(want, axis=1), 1e-30)
        assert err.max() < 1e-5, err.max()
    # central differences of the FP64 residual along random directions
    h = 1e-4
    for trial in range(3):
        vp = rng.normal(size=(F, 6)) * np.array([1e-2] * 3 + [1e-1] * 3)
        vx = rng.normal(size=(P, 3)) * 1e-1
        fd = ((_oracle_e(prob, h * vp, h * vx) - _oracle_e(prob, -h * vp, -h * vx)) * G).sum() / (2 * h)
        ad = (gpose * vp).sum() + (gpoint * vx).sum()
        assert abs(ad - fd) <= 1e-5 * max(abs(fd), np.abs(gpose * vp).sum() + np.abs(gpoint * vx).sum())
    lin.close()


def test_forward_moves_with_increments(gpu_ctx):
    import torch
    prob = _problem()
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P = len(prob.frames), len(prob.points)
    rng = np.random.default_rng(1)
    dp = rng.normal(size=(F, 6)) * 1e-3
    dx = rng.normal(size=(P, 3)) * 1e-3
    e = reprojection(torch.from_numpy(dp).cuda(), torch.from_numpy(dx).cuda(), lin,
                     (prob.points, prob.frames, prob.cams)).cpu().numpy()
    re = _oracle_e(prob, dp, dx)
    err = np.linalg.norm(e - re, axis=1) / np.maximum(np.linalg.norm(re, axis=1), 1e-9)
    assert err.max() < 1e-5
    lin.close()


def test_backward_after_relinearization_raises(gpu_ctx):
    """Two forwards on one BALinearizer, then the first one's backward: its
    Jacobians were overwritten by the second forward, so backward refuses
    instead of returning another state's gradient."""
    import torch
    prob = _problem()
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P = len(prob.frames), len(prob.points)
    d1 = torch.zeros((F, 6), dtype=torch.float64, device="cuda", requires_grad=True)
    x1 = torch.zeros((P, 3), dtype=torch.float64, device="cuda", requires_grad=True)
    e1 = reprojection(d1, x1, lin, (prob.points, prob.frames, prob.cams))
    d2 = torch.full((F, 6), 1e-3, dtype=torch.float64, device="cuda", requires_grad=True)
    e2 = reprojection(d2, x1, lin, (prob.points, prob.frames, prob.cams))
    with pytest.raises(RuntimeError, match="relinearized"):
        (e1.sum() + e2.sum()).backward()
    # the latest forward's backward still works
    x3 = torch.zeros((P, 3), dtype=torch.float64, device="cuda", requires_grad=True)
    e3 = reprojection(d1.detach().requires_grad_(), x3, lin, (prob.points, prob.frames, prob.cams))
    e3.sum().backward()
    assert torch.isfinite(x3.grad).all()
    lin.close()


def test_adjoint_at_150k_observations(gpu_ctx):
    """The adjoint at the BA linearization configuration's size (10 keyframes
    x 3 cameras, 20k points, ~150k observations) against the FP64 analytic
    J^T g."""
    import torch
    prob = synth.ba_problem(seed=30, n_kf=10, n_points=20000, target_obs=150000)
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P, M = len(prob.frames), len(prob.points), len(prob.obs_pt)
    dpose = torch.zeros((F, 6), dtype=torch.float64, device="cuda", requires_grad=True)
    dpoint = torch.zeros((P, 3), dtype=torch.float64, device="cuda", requires_grad=True)
    e = reprojection(dpose, dpoint, lin, (prob.points, prob.frames, prob.cams))
    G = np.random.default_rng(7).normal(size=(M, 2))
    (e * torch.from_numpy(G).float().cuda()).sum().backward()
    _, _, _, Jp, Jx = oracle.ba_linearize(prob)
    want_pose = np.zeros((F, 6))
    want_point = np.zeros((P, 3))
    np.add.at(want_pose, prob.obs_frame, np.einsum("mij,mi->mj", Jp, G))
    np.add.at(want_point, prob.obs_pt, np.einsum("mij,mi->mj", Jx, G))
    for got, want in ((dpose.grad.cpu().numpy(), want_pose), (dpoint.grad.cpu().numpy(), want_point)):
        err = np.linalg.norm(got - want, axis=1) / np.maximum(np.linalg.norm(want, axis=1), 1e-30)
        print(f"adjoint 150k: max rel err {err.max():.2e}", flush=True)
        assert err.max() < 1e-5
    lin.close()


@pytest.mark.parametrize("dtype", ["float32", "float64"])
def test_increments_on_the_device(gpu_ctx, dtype):
    """Increments applied on the device against the host's: full tensors of
    both types, strided ones, one frame's increment zero; broadcast and
    half-precision increments still take the host's way."""
    import torch
    prob = _problem()
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P = len(prob.frames), len(prob.points)
    dt = getattr(torch, dtype)
    rng = np.random.default_rng(2)
    dp = torch.from_numpy(rng.normal(size=(F, 6)) * 1e-2).to(dt).cuda()
    dp[1] = 0
    dx = torch.from_numpy(rng.normal(size=(P, 3)) * 1e-2).to(dt).cuda()
    state = (prob.points, prob.frames, prob.cams)

    def check(a, b):
        e = reprojection(a, b, lin, state)
        assert e.shape == (lin.M, 2) and e.is_contiguous()
        re = _oracle_e(prob, a.double().cpu().numpy(), b.double().cpu().numpy())
        err = np.linalg.norm(e.cpu().numpy() - re, axis=1) / np.maximum(np.linalg.norm(re, axis=1), 1e-9)
        assert err.max() < 1e-5
        pts, frs = apply_increments(prob.points, prob.frames, a.double().cpu().numpy(), b.double().cpu().numpy())
        got_pts, got_frs = lin.get_state()
        np.testing.assert_array_equal(got_pts, pts)
        assert np.abs(got_frs - frs * np.where(frs[:, 3:4] < 0, np.array([[-1.] * 4 + [1.] * 3]), 1.0)).max() < 1e-13

    check(dp, dx)
    check(dp.repeat(1, 2)[:, ::2], dx.t().contiguous().t())
    check(dp, dx[:1])                     # one increment for every point
    if dtype == "float32":
        check(dp.half(), dx)
    lin.close()


@pytest.mark.parametrize("n_kf,n_points,obs", [(1, 40, 40), (2, 900, 1500), (1, 4200, 4200)])
def test_pose_adjoint_sizes(gpu_ctx, n_kf, n_points, obs):
    """Frames of fewer observations than the adjoint's workgroup has threads,
    and of a little more than one round of it.  Bound: sums of n float32
    products in any order, n eps sum |J^T g|."""
    import torch
    prob = synth.ba_problem(seed=50 + n_kf, n_kf=n_kf, n_points=n_points, target_obs=obs)
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P, M = len(prob.frames), len(prob.points), len(prob.obs_pt)
    z = lambda n, k: torch.zeros((n, k), dtype=torch.float32, device="cuda", requires_grad=True)
    dpose, dpoint = z(F, 6), z(P, 3)
    e = reprojection(dpose, dpoint, lin, (prob.points, prob.frames, prob.cams))
    G = np.random.default_rng(1).normal(size=(M, 2)).astype(np.float32)
    (e * torch.from_numpy(G).cuda()).sum().backward()
    J = lin.results()[3].astype(np.float64)
    terms = np.einsum("mij,mi->mj", J, G.astype(np.float64))
    want, mag = np.zeros((F, 6)), np.zeros((F, 6))
    np.add.at(want, prob.obs_frame, terms)
    np.add.at(mag, prob.obs_frame, np.einsum("mij,mi->mj", np.abs(J), np.abs(G).astype(np.float64)))
    assert (np.abs(dpose.grad.cpu().numpy() - want) <= M * 2.0 ** -24 * mag + 1e-30).all()
    lin.close()


def test_negated_views(gpu_ctx):
    """Tensors whose negation is a flag on shared memory (what the imaginary
    part of a conjugated complex tensor is): increments and an incoming
    gradient of that kind give what their values in memory of their own give."""
    import torch
    prob = _problem()
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P = len(prob.frames), len(prob.points)
    rng = np.random.default_rng(4)
    dp = torch.from_numpy(rng.normal(size=(F, 6)) * 1e-2).float().cuda()
    dx = torch.from_numpy(rng.normal(size=(P, 3)) * 1e-2).float().cuda()
    g = torch.from_numpy(rng.normal(size=(lin.M, 2))).float().cuda()
    out = []
    for neg in (torch._neg_view, torch.neg):
        a, b = neg(dp).requires_grad_(), neg(dx).requires_grad_()
        assert a.is_neg() == (neg is torch._neg_view)
        e = reprojection(a, b, lin, (prob.points, prob.frames, prob.cams))
        out.append((e, *torch.autograd.grad(e, (a, b), neg(g))))
    for x, y in zip(*out):
        np.testing.assert_array_equal(x.detach().cpu().numpy(), y.detach().cpu().numpy())
    lin.close()


@pytest.mark.parametrize("F,M,shape", [(21, 3000, "1024, 1"), (22, 3000, "256, 1"), (42, 500001, "256, 1"),
                                       (43, 500000, "256, 1"), (43, 500001, "256, 3"), (128, 500001, "256, 3"),
                                       (129, 500001, "256, 6"), (300, 900, "256, 1")])
def test_pose_adjoint_shapes(gpu_ctx, F, M, shape):
    """Both sides of every line between the pose adjoint's launch shapes, the
    last frame without observations.  Bound as above, n the frame's own
    observations and the roundings of a term."""
    import torch
    rng = np.random.default_rng(F + M)
    P = M // 8
    fr = rng.integers(0, F - 1, M)
    lin = BALinearizer(M, P, F, 1, gpu_ctx)
    lin.set_observations(rng.uniform(0, 600, (M, 2)), np.sort(rng.integers(0, P, M)), fr, np.zeros(M), np.ones(M))
    lin.set_state(np.c_[rng.uniform(-2, 2, (P, 2)), rng.uniform(3, 9, P)], np.tile([0, 0, 0, 1., 0, 0, 0], (F, 1)),
                  [[700, 700, 640, 360, 0, 0, 0, 1., 0, 0, 0, 2.]])
    G = rng.normal(size=(M, 2)).astype(np.float32)
    g = torch.from_numpy(G).cuda()
    pose, point = torch.full((F, 6), 9.0, device="cuda"), torch.empty((P, 3), device="cuda")
    lin.ctx.use_torch_stream()
    lin.linearize()
    kernel = f"k_ba_pose_adj<{shape}>"
    names = device_events(lambda: lin.adjoint_dev(g.data_ptr(), pose.data_ptr(), point.data_ptr()), [kernel])
    assert {n.split("(")[0] for n in names if "k_ba_pose_adj" in n} == {"void mcv::" + kernel}
    J = lin.read(4, 12).astype(np.float64).reshape(2, 6, M)
    G = G.T.astype(np.float64)
    got = pose.cpu().numpy()
    n = np.bincount(fr, minlength=F)
    for c in range(6):
        want = np.bincount(fr, J[0, c] * G[0] + J[1, c] * G[1], F)
        mag = np.bincount(fr, np.abs(J[0, c] * G[0]) + np.abs(J[1, c] * G[1]), F)
        assert (np.abs(got[:, c] - want) <= (n + 2) * 2.0 ** -24 * mag + 1e-30).all()
    lin.close()


def test_set_state_increments_checks_its_tensors(gpu_ctx):
    """What the device would read past or misread is refused before anything
    is enqueued; strided tensors give what dense ones give."""
    import torch
    prob = _problem()
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    F, P = len(prob.frames), len(prob.points)
    state = (prob.points, prob.frames, prob.cams)
    dp, dx = torch.full((F, 6), 1e-2, device="cuda"), torch.full((P, 3), 1e-2, device="cuda")
    before = lin.get_state()
    for a, b in ((dp[:-1], dx), (dp, dx[:-1]), (dp, dx[:1]), (dp.half(), dx), (dp, dx.int()), (dp.cpu(), dx),
                 (dp, dx.cpu()), (dp.flatten(), dx), (dp, dx[:, :2])):
        with pytest.raises(ValueError):
            lin.set_state_increments(*state, a, b)
    with pytest.raises(ValueError):
        lin.set_state_increments(prob.points[:-1], prob.frames, prob.cams, dp, dx)
    for x, y in zip(before, lin.get_state()):
        np.testing.assert_array_equal(x, y)
    lin.set_state_increments(*state, dp, dx)
    want = lin.get_state()
    lin.set_state_increments(*state, dp.repeat(1, 2)[:, ::2], dx.t().contiguous().t())
    for x, y in zip(want, lin.get_state()):
        np.testing.assert_array_equal(x, y)
    lin.close()
