"""Local bundle adjustment on the GPU against the FP64 oracle: the
pose-only linearization mode, the Schur complement with stereo edges, fixed
points and inactive edges against the dense damped normal equations, the
robust chi2 reduction, ten Levenberg-Marquardt iterations of
PoseEstimation::BoundleAdjustment with its chi2 outlier pass, and the four
rounds of PoseEstimation::PoseOptimization
(core/optimization_algorithm_levenberg.cpp:56-159, core/block_solver.hpp:
315-449, include/PoseEstimation.hpp:35-119, src/PoseEstimation.cpp:45-151)."""
import numpy as np
import pytest

import oracle
from kernel_check import device_events
from lm_check import dense_schur, dense_system
from mcvslam_amd import BALinearizer, synth
from mcvslam_amd.ba import bundle_adjustment, local_ba_linearizer, pose_optimization

pytestmark = pytest.mark.gpu


def _lin(lp, ctx):
    return local_ba_linearizer(lp.mono, lp.stereo, lp.point_fixed, ctx=ctx)


def test_pose_only_mode_writes_all_but_j_point(gpu_ctx):
    prob = synth.ba_problem(seed=70, n_kf=4, n_points=2000, target_obs=15000)
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    shifted = prob.points + 0.1
    b.linearize()
    full_a = b.read()
    b.set_state(shifted, prob.frames, prob.cams)
    b.linearize()
    full_b = b.read()
    b.set_state(prob.points, prob.frames, prob.cams)
    b.linearize()
    b.set_state(shifted, prob.frames, prob.cams)
    b.linearize(mode=BALinearizer.POSE_ONLY)
    pose_b = b.read()
    np.testing.assert_array_equal(pose_b[:16], full_b[:16])
    np.testing.assert_array_equal(pose_b[16:], full_a[16:])     # J_point planes untouched
    assert not np.array_equal(full_a[16:], full_b[16:])
    # the stereo edge likewise: J_point rows are planes 23..31
    sp = synth.stereo_problem(seed=70, n_kf=4, n_points=2000, target_obs=3000)
    b2 = BALinearizer.from_problem(synth.ba_problem(seed=70, n_kf=4, n_points=2000, target_obs=5000), ctx=gpu_ctx)
    b2.set_stereo(sp.obs, sp.obs_pt, sp.obs_frame, sp.obs_isig, sp.cam)
    b2.linearize_stereo()
    e_a, _, _, jp_a, jx_a = b2.stereo_results()
    b2.set_state(sp.points + 0.1, sp.frames, b2_cams(sp))
    b2.set_stereo(sp.obs, sp.obs_pt, sp.obs_frame, sp.obs_isig, sp.cam)
    b2.linearize_stereo(mode=BALinearizer.POSE_ONLY)
    e_b, _, _, jp_b, jx_b = b2.stereo_results()
    np.testing.assert_array_equal(jx_b, jx_a)
    assert not np.array_equal(e_a, e_b) and not np.array_equal(jp_a, jp_b)


def b2_cams(sp):
    return synth.ba_problem(seed=70, n_kf=4, n_points=2000, target_obs=5000).cams


@pytest.mark.parametrize("robust", [True, False])
def test_schur_with_stereo_fixed_points_and_levels_vs_dense(gpu_ctx, robust):
    lp = synth.local_ba_problem(seed=71, n_kf=5, n_points=800, target_obs=8000, stereo_frac=0.9)
    rng = np.random.default_rng(3)
    am = (rng.random(len(lp.mono.obs_pt)) > 0.1).astype(np.uint8)
    ast = (rng.random(len(lp.stereo.obs_pt)) > 0.1).astype(np.uint8)
    lin = _lin(lp, gpu_ctx)
    assert lin.Ms > 50 and lp.point_fixed.sum() > 10
    lin.set_active(am, ast)
    lin.set_robust(robust)
    lin.linearize()
    lin.linearize_stereo()
    H, b, lam, free_f, free_p = dense_system(lp, lp.mono.points, lp.mono.frames, active_m=am, active_s=ast,
                                             robust=robust)
    S_ref, bs_ref = dense_schur(H, b, lam, 6 * len(free_f))
    S, bs = lin.schur(lam)
    es = np.linalg.norm(S - S_ref) / np.linalg.norm(S_ref)
    eb = np.linalg.norm(bs - bs_ref) / np.linalg.norm(bs_ref)
    print(f"Schur with stereo/fixed points/levels (robust={robust}): rel err S {es:.2e}, b {eb:.2e}", flush=True)
    assert es < 1e-5 and eb < 1e-4


@pytest.mark.parametrize("n_kf,n_points,obs,off", [(2, 20, 40, 0), (2, 260, 513, 0), (12, 150, 1030, 600),
                                                   (21, 80, 1100, 0)])
def test_schur_chunks_vs_dense(gpu_ctx, n_kf, n_points, obs, off):
    """The Schur complement at the edges of its work division: 1, 11 and 20
    free frames (18, 1 and 1 threads per frame sum), edge counts on both sides
    of the 512-edge chunks, a chunk whose edges are all inactive, points with
    more than 8 edges and frames.  Tolerances as the dense comparison above."""
    lp = synth.local_ba_problem(seed=75, n_kf=n_kf, n_points=n_points, target_obs=obs, stereo_frac=0.6)
    lin = _lin(lp, gpu_ctx)
    am = np.ones(lin.M, np.uint8)
    am[:off] = 0
    lin.set_active(am)
    lin.linearize()
    lin.linearize_stereo()
    H, b, _, free_f, _ = dense_system(lp, lp.mono.points, lp.mono.frames, active_m=am)
    for lam in (1e2, 1e4):
        S_ref, bs_ref = dense_schur(H, b, lam, 6 * len(free_f))
        S, bs = lin.schur(lam)
        assert np.linalg.norm(S - S_ref) < 1e-5 * np.linalg.norm(S_ref)
        assert np.linalg.norm(bs - bs_ref) < 1e-4 * np.linalg.norm(bs_ref)
    np.testing.assert_array_equal(lin.schur(1e4)[0], S)     # summation orders are fixed
    lin.close()


def test_robust_chi2_vs_oracle(gpu_ctx):
    lp = synth.local_ba_problem(seed=73, n_kf=6, n_points=3000, target_obs=30000, stereo_frac=0.8)
    lin = _lin(lp, gpu_ctx)
    rng = np.random.default_rng(4)
    am = (rng.random(len(lp.mono.obs_pt)) > 0.2).astype(np.uint8)
    for robust in (True, False):
        for act in (None, am):
            lin.set_robust(robust)
            lin.set_active(act, None)
            lin.linearize(residual_only=True)
            lin.linearize_stereo(residual_only=True)
            got = lin.robust_chi2()
            want = oracle.ba_robust_chi2(lp.mono, lp.stereo, robust=robust, active=act)
            assert abs(got - want) < 1e-5 * want, (robust, act is None, got, want)


def _oracle_chi2(lp, pts, frs):
    m = lp.mono
    prob = synth.BAProblem(m.obs_uv, m.obs_pt, m.obs_frame, m.obs_cam, m.obs_level, m.obs_isig, pts, frs, m.cams,
                           m.frame_fixed)
    chi2 = oracle.ba_linearize(prob)[1]
    s = lp.stereo
    schi2 = oracle.ba_stereo_linearize(s.obs, s.obs_pt, s.obs_frame, s.obs_isig, pts, frs, s.cam)[1]
    return chi2, schi2


def test_bundle_adjustment_10_iterations_vs_fp64_oracle(gpu_ctx):
    """The BA linearization configuration (10 keyframes x 3 cameras, 20k
    points, ~150k observations) with LEFT stereo edges, keyframe 0 and a
    tenth of the points fixed, from a perturbed state: ten LM iterations on
    the GPU (FP32 linearization and Schur, FP64 Cholesky) against the FP64
    oracle LM, then FilterCallBack_Chi2."""
    lp = synth.local_ba_problem(seed=72, n_kf=10, n_points=20000, target_obs=150000, stereo_frac=0.5)
    lin = _lin(lp, gpu_ctx)
    res = bundle_adjustment(lin, 10)
    opts, ofrs, ost, on, _ = oracle.ba_lm(lp.mono, lp.stereo, iterations=10, point_fixed=lp.point_fixed)
    print("gpu   :", np.array2string(res.stats, precision=6), flush=True)
    print("oracle:", np.array2string(ost, precision=6), flush=True)
    assert res.iterations == on == 10
    rel = np.abs(res.stats[:, :2] - ost[:, :2]) / ost[:, :2]
    print(f"chi2 trajectory max rel diff {rel.max():.2e}", flush=True)
    assert rel.max() < 1e-4
    assert res.stats[-1, 1] < 0.9 * res.stats[0, 0]
    pts, frs = res.points, res.frames
    dt = np.abs(frs[:, 4:] - ofrs[:, 4:]).max()
    dq = min(np.abs(frs[:, :4] - ofrs[:, :4]).max(), np.abs(frs[:, :4] + ofrs[:, :4]).max())
    dp = np.abs(pts - opts).max(1)
    print(f"state: max |dt| {dt:.2e} m, max |dq| {dq:.2e}, points p99 {np.percentile(dp, 99):.2e} m, "
          f"max {dp.max():.2e} m", flush=True)
    assert dt < 1e-4 and dq < 1e-5 and np.percentile(dp, 99) < 1e-3
    # FilterCallBack_Chi2 at the optimized states
    chi2, schi2 = _oracle_chi2(lp, opts, ofrs)
    thr = 5.991
    for got, c in ((res.outliers_mono, chi2), (res.outliers_stereo, schi2)):
        want = (c.astype(np.float32) >= np.float32(thr)).astype(np.uint8)
        far = np.abs(c - thr) > 1e-3 * thr
        np.testing.assert_array_equal(got[far], want[far])
        assert 0 < got.sum() < len(got)


def _pose_problem(seed):
    """PoseOptimization's graph: one keyframe free, every point fixed, its
    mono and stereo edges."""
    lp = synth.local_ba_problem(seed=seed, n_kf=3, n_points=3000, target_obs=20000, stereo_frac=0.8,
                                perturb_pose=0.02, fixed_point_frac=0.0)
    m, s = lp.mono, lp.stereo
    km, ks = m.obs_frame == 2, s.obs_frame == 2
    mono = synth.BAProblem(m.obs_uv[km], m.obs_pt[km], m.obs_frame[km], m.obs_cam[km], m.obs_level[km],
                           m.obs_isig[km], lp.true_points.copy(), m.frames, m.cams, np.array([1, 1, 0], np.int32))
    stereo = synth.StereoProblem(s.obs[ks], s.obs_pt[ks], s.obs_frame[ks], s.obs_isig[ks], mono.points, mono.frames,
                                 s.cam)
    return mono, stereo, np.ones(len(mono.points), np.int32)


def test_pose_optimization_rounds_vs_oracle(gpu_ctx):
    mono, stereo, pfix = _pose_problem(74)
    lin = local_ba_linearizer(mono, stereo, pfix, ctx=gpu_ctx)
    res = pose_optimization(lin)
    # the oracle runs the same four rounds
    am, ast = np.ones(len(mono.obs_pt), np.uint8), np.ones(len(stereo.obs_pt), np.uint8)
    pts, frs = mono.points, mono.frames
    robust = True
    n_init = len(am) + len(ast)
    lp = synth.LocalBAProblem(mono, stereo, pfix, None, None)
    for it in range(4):
        pts, frs, _, _, _ = oracle.ba_lm(mono, stereo, iterations=15, point_fixed=pfix, active=am, sactive=ast,
                                         robust=robust, points=pts, frames=frs)
        chi2, schi2 = _oracle_chi2(lp, pts, frs)
        bm = (am == 1) & (chi2.astype(np.float32) >= np.float32(5.991))
        bs = (ast == 1) & (schi2.astype(np.float32) >= np.float32(5.991))
        am[bm] = 0
        ast[bs] = 0
        if it == 2:
            robust = False
        if n_init - bm.sum() - bs.sum() < 10:
            break
    assert res.frames is not None
    dt = np.abs(res.frames[2, 4:] - frs[2, 4:]).max()
    dq = min(np.abs(res.frames[2, :4] - frs[2, :4]).max(), np.abs(res.frames[2, :4] + frs[2, :4]).max())
    nd = int((res.active_mono != am).sum() + (res.active_stereo != ast).sum())
    print(f"pose optimization: |dt| {dt:.2e}, |dq| {dq:.2e}, level disagreements {nd} of {n_init}, "
          f"inliers {res.inliers}", flush=True)
    assert dt < 1e-5 and dq < 1e-6
    assert nd <= max(2, n_init // 1000)
    assert (am == 0).sum() > 0


@pytest.mark.parametrize("n_kf,n_points,obs,stereo_frac", [(1, 40, 25, 0.9), (1, 1500, 1024, 0.0), (3, 900, 2049, 0.9),
                                                           (1, 9000, 7000, 0.5)])
@pytest.mark.parametrize("robust", [True, False])
def test_single_pose_route_vs_oracle_and_general_route(gpu_ctx, n_kf, n_points, obs, stereo_frac, robust):
    """One free keyframe, every point fixed: the one-launch trials against the
    oracle LM and against the general route, which the same problem takes when
    a point without edges is left free.  Edge counts around the workgroup's
    1024 threads, other keyframes fixed, inactive edges.  Tolerances as
    test_pose_optimization_rounds_vs_oracle, whose sums are as wide."""
    lp = synth.local_ba_problem(seed=76, n_kf=n_kf, n_points=n_points, target_obs=obs, stereo_frac=stereo_frac,
                                fixed_point_frac=1.0, perturb_pose=0.0)
    mono, stereo = lp.mono, lp.stereo if len(lp.stereo.obs_pt) else None
    free = n_kf - 1
    mono.frame_fixed = np.ones(n_kf, np.int32)
    mono.frame_fixed[free] = 0
    f = oracle.se3_oplus(mono.frames[free], np.random.default_rng(5).normal(0, 0.01, 6))
    mono.frames[free] = f
    mono.points = np.concatenate([mono.points, [[0.0, 0.0, 5.0]]])       # seen by no edge
    am = (np.random.default_rng(6).random(len(mono.obs_pt)) > 0.1).astype(np.uint8)
    out = []
    for last in (1, 0):
        pfix = np.ones(len(mono.points), np.int32)
        pfix[-1] = last
        lin = local_ba_linearizer(mono, stereo, pfix, ctx=gpu_ctx)
        lin.set_active(am)
        lin.set_robust(robust)
        stats, n = lin.optimize(6)
        out.append((stats, lin.get_state()[1], lin.outliers(stereo=stereo is not None)))
        lin.close()
    _, frs, ost, _, _ = oracle.ba_lm(mono, stereo, iterations=6, point_fixed=np.ones(len(mono.points), np.int32),
                                     active=am, robust=robust)
    for stats, got, _ in out:
        assert np.abs(got[free, 4:] - frs[free, 4:]).max() < 1e-5
        assert np.abs(got[free, :4] - frs[free, :4]).max() < 1e-6
        np.testing.assert_array_equal(np.delete(got, free, 0), np.delete(mono.frames, free, 0))
        assert abs(stats[0, 0] - ost[0, 0]) < 1e-5 * ost[0, 0]
        assert abs(stats[-1, 1] - ost[-1, 1]) < 1e-5 * ost[-1, 1]
    for a, b in zip(out[0][2], out[1][2]):
        if a is not None:
            assert (a != b).sum() <= max(2, len(a) // 1000)


def test_single_pose_more_iterations_than_one_launch(gpu_ctx):
    """A first lambda so large that the steps stay small for some 20
    iterations: more than one launch of the one-frame optimizer runs (16).
    Against the general route, which the same problem takes when a point
    without edges is left free; tolerances as above."""
    lp = synth.local_ba_problem(seed=77, n_kf=1, n_points=700, target_obs=500, stereo_frac=0.5, fixed_point_frac=1.0,
                                perturb_pose=0.0)
    mono = lp.mono
    mono.frame_fixed = np.zeros(1, np.int32)
    mono.frames[0] = oracle.se3_oplus(mono.frames[0], np.random.default_rng(5).normal(0, 0.01, 6))
    mono.points = np.concatenate([mono.points, [[0.0, 0.0, 5.0]]])       # seen by no edge
    out = []
    for last in (1, 0):
        pfix = np.ones(len(mono.points), np.int32)
        pfix[-1] = last
        lin = local_ba_linearizer(mono, lp.stereo, pfix, ctx=gpu_ctx)
        stats, n = lin.optimize(40, tau=1e8)
        out.append((stats, n, lin.get_state()[1]))
        lin.close()
    assert out[0][1] > 17 and out[1][1] > 17
    k = 17                                # the iterations around the second launch's start
    np.testing.assert_allclose(out[0][0][:k + 1, :3], out[1][0][:k + 1, :3], rtol=1e-3)
    assert np.abs(out[0][2][0, 4:] - out[1][2][0, 4:]).max() < 1e-5
    assert np.abs(out[0][2][0, :4] - out[1][2][0, :4]).max() < 1e-6


def test_schur_stays_readable_after_a_refused_call(gpu_ctx):
    """Stereo edges set but not linearized: the Schur complement is refused and
    the last one is still what is read; after the linearization it is theirs."""
    import ctypes
    from mcvslam_amd import MCVError
    from mcvslam_amd._native import lib
    lp = synth.local_ba_problem(seed=78, n_kf=5, n_points=300, target_obs=3000, stereo_frac=0.5)
    lin = BALinearizer.from_problem(lp.mono, ctx=gpu_ctx)
    lin.linearize()
    S, bs = lin.schur(1e3)
    s = lp.stereo
    lin.set_stereo(s.obs, s.obs_pt, s.obs_frame, s.obs_isig, s.cam)
    with pytest.raises(MCVError):
        lin.schur(1e3)
    got, gb, n = np.zeros_like(S), np.zeros_like(bs), ctypes.c_int32()
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    assert lib().mcv_ba_read_schur(lin.h, ptr(got), ptr(gb), ctypes.byref(n)) == 0 and n.value == len(bs)
    np.testing.assert_array_equal(got, S)
    np.testing.assert_array_equal(gb, bs)
    lin.linearize_stereo()
    assert not np.array_equal(lin.schur(1e3)[0], S)
    lin.close()


def _many_frames(n_kf, n_points, seen, seed):
    """Keyframes side by side before a wall of points.  Every point is seen by
    keyframes 0, 1 and 2 (pairs with more shared points than one chunk of
    items) and by `seen` others, some of them with two cameras."""
    rng = np.random.default_rng(seed)
    q = rng.normal(0, 0.02, (n_kf, 4)) + [0, 0, 0, 1.0]
    frames = np.c_[q / np.linalg.norm(q, axis=1)[:, None], rng.uniform(-1, 1, (n_kf, 2)), rng.uniform(-0.3, 0.3, n_kf)]
    points = np.c_[rng.uniform(-2, 2, (n_points, 2)), rng.uniform(4, 8, n_points)]
    cams = np.array([[500, 500, 320, 240, 0, 0, 0, 1.0, 0.1 * k, 0, 0, 2.4] for k in range(2)])
    rows = [(p, f, c) for p in range(n_points)
            for f in np.r_[0, 1, 2, rng.choice(np.arange(3, n_kf), seen, replace=False)]
            for c in range(1 + (rng.random() < 0.2))]
    pt, fr, cam = np.array(rows).T
    R = _rotations(frames)
    x = np.einsum("mij,mj->mi", R[fr], points[pt]) + frames[fr, 4:]
    x[:, 0] += 0.1 * cam
    uv = (500 * x[:, :2] / x[:, 2:] + [320, 240] + rng.normal(0, 1.0, (len(pt), 2))).astype(np.float32)
    fixed = np.zeros(n_kf, np.int32)
    fixed[-1] = 1
    return synth.BAProblem(uv, pt.astype(np.int32), fr.astype(np.int32), cam.astype(np.int32), np.zeros(len(pt), np.int32),
                           np.ones(len(pt), np.float32), points, frames, cams, fixed)


def _rotations(frames):
    x, y, z, w = frames[:, :4].T
    return np.array([[1 - 2 * (y * y + z * z), 2 * (x * y - z * w), 2 * (x * z + y * w)],
                     [2 * (x * y + z * w), 1 - 2 * (x * x + z * z), 2 * (y * z - x * w)],
                     [2 * (x * z - y * w), 2 * (y * z + x * w), 1 - 2 * (x * x + y * y)]]).transpose(2, 0, 1)


def _check_schur_fp64(lin, prob):
    """The Schur complement of a linearized _many_frames problem against the
    FP64 sums over its points; tolerances as the dense comparisons above."""
    n_kf = len(prob.frames)
    e, _, w, Jp, Jx = oracle.ba_linearize(prob)
    W = w * prob.obs_isig
    m = 6 * (n_kf - 1)
    for lam in (1e2, 1e4):
        S_ref, bs_ref = lam * np.eye(m), np.zeros(m)
        for p in range(len(prob.points)):
            i = np.nonzero(prob.obs_pt == p)[0]
            B, r, ww = Jx[i].reshape(-1, 3), e[i].ravel(), W[i].repeat(2)[:, None]
            A = np.zeros((2 * len(i), n_kf, 6))
            A[np.arange(2 * len(i)), prob.obs_frame[i].repeat(2)] = Jp[i].reshape(-1, 6)
            used = np.unique(prob.obs_frame[i])
            used = used[used < n_kf - 1]
            A = A[:, used].reshape(2 * len(i), -1)
            D = (ww * B).T @ B + lam * np.eye(3)
            C, bl = (ww * A).T @ B, -(ww * B).T @ r
            at = (6 * used[:, None] + np.arange(6)).ravel()
            S_ref[np.ix_(at, at)] += (ww * A).T @ A - C @ np.linalg.solve(D, C.T)
            bs_ref[at] += -(ww * A).T @ r - C @ np.linalg.solve(D, bl)
        S, bs = lin.schur(lam)
        assert np.linalg.norm(S - S_ref) < 1e-5 * np.linalg.norm(S_ref)
        assert np.linalg.norm(bs - bs_ref) < 1e-4 * np.linalg.norm(bs_ref)
        np.testing.assert_array_equal(lin.schur(lam)[0], S)


@pytest.mark.parametrize("n_kf", [65, 66, 71, 131])
def test_schur_many_frames_vs_fp64(gpu_ctx, n_kf):
    """64 free keyframes and more: masks of more than one 64-bit word."""
    prob = _many_frames(n_kf, 700, 8, n_kf)
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    lin.linearize()
    _check_schur_fp64(lin, prob)
    lin.close()


def test_schur_frame_sums_of_many_chunks(gpu_ctx):
    """1000 free keyframes with 2M mono and 0.6M stereo edges: a row of frame
    sums per chunk would take 550 MB, so workgroups take several chunks, mono
    and stereo ones among them.  Every point is fixed, so S is H_pp + lambda I.
    Bound: sums of n FP32 products in any order.  What stays allocated: 116
    bytes an edge of lists and entry rows, S, at most 256 MiB of frame sums."""
    import torch
    from mcvslam_amd import Context
    ctx = Context(0)
    F, P, M, Ms = 1000, 5000, 2_000_000, 600_000
    rng = np.random.default_rng(79)
    fr, sfr = rng.integers(0, F, M), rng.integers(0, F, Ms)
    lin = BALinearizer(M, P, F, 1, ctx)
    lin.set_observations(rng.uniform(0, 640, (M, 2)), np.sort(rng.integers(0, P, M)), fr, np.zeros(M), np.ones(M))
    cam = [500, 500, 320, 240, 0, 0, 0, 1.0, 0, 0, 0, 2.4]
    lin.set_state(np.c_[rng.uniform(-1, 1, (P, 2)), rng.uniform(4, 8, P)], np.tile([0, 0, 0, 1.0, 0, 0, 0], (F, 1)), [cam])
    obs = rng.uniform(0, 640, (Ms, 3))
    lin.set_stereo(obs, rng.integers(0, P, Ms), sfr, np.ones(Ms), [500, 500, 320, 240, 50, 2.8])
    lin.set_fixed(np.zeros(F))
    lin.set_point_fixed(np.ones(P))
    lin.linearize()
    lin.linearize_stereo()
    ctx.synchronize()
    free = torch.cuda.mem_get_info()[0]
    S, bs = lin.schur(10.0)
    assert free - torch.cuda.mem_get_info()[0] < 116 * (M + Ms) + 144e6 + (256 << 20) + 40e6
    e, _, w, Jp, _ = lin.results()
    se, _, sw, sJp, _ = lin.stereo_results()
    f64 = lambda a: np.asarray(a, np.float64)
    blocks = S.reshape(F, 6, F, 6)
    got = blocks[np.arange(F), :, np.arange(F)]
    n = np.bincount(fr, minlength=F) * 2 + np.bincount(sfr, minlength=F) * 3
    for i in range(6):
        for j in range(i, 7):
            want, mag = np.zeros(F), np.zeros(F)
            for J, r, W, f in ((Jp, e, w, fr), (sJp, se, sw, sfr)):
                t = f64(W)[:, None] * f64(J[:, :, i]) * (f64(J[:, :, j]) if j < 6 else -f64(r))
                want += np.bincount(f, t.sum(1), F)
                mag += np.bincount(f, np.abs(t).sum(1), F)
            if j == i:
                want += 10.0
            x = got[:, i, j] if j < 6 else bs.reshape(F, 6)[:, i]
            assert (np.abs(x - want) <= (n + 4) * 2.0 ** -24 * (mag + 10.0)).all(), (i, j)
    blocks[np.arange(F), :, np.arange(F)] = 0
    assert not S.any()
    lin.close()
    ctx.close()


@pytest.mark.parametrize("n_kf,fetched", [(126, False), (127, True), (160, True)])
def test_schur_windows_of_cut_pairs(gpu_ctx, n_kf, fetched):
    """125 free keyframes and fewer: the windows of every keyframe pair come to
    the host in one table; more: those of the pairs whose items are cut into
    chunks alone (the pairs of keyframes 0, 1 and 2 here)."""
    prob = _many_frames(n_kf, 700, 8, n_kf)
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    lin.linearize()

    def build():
        lin.set_active(np.ones(lin.M, np.uint8))          # the lists are built anew
        lin.schur(1e2)

    names = device_events(build, ["k_sb_blocks"] + ["k_sb_windows"] * fetched)
    assert any("k_sb_windows" in n for n in names) == fetched
    _check_schur_fp64(lin, prob)
    lin.close()


def _one_frame(n_edges, n_cams, n_stereo, seed):
    """One keyframe before a wall of fixed points, the last one unseen: exactly
    n_edges mono edges over n_cams cameras and n_stereo stereo edges, from a
    perturbed pose."""
    rng = np.random.default_rng(seed)
    P = max(-(-n_edges // n_cams), n_stereo) + 1
    points = np.c_[rng.uniform(-2, 2, (P, 2)), rng.uniform(4, 8, P)]
    cams = np.array([[500, 500, 320, 240, 0, 0, 0, 1.0, 0.05 * k, -0.02 * k, 0, 2.4] for k in range(n_cams)])
    pt, cam = np.repeat(np.arange(P - 1), n_cams)[:n_edges], np.tile(np.arange(n_cams), P - 1)[:n_edges]
    x = points[pt] + cams[cam, 8:11]
    uv = 500 * x[:, :2] / x[:, 2:] + [320, 240] + rng.normal(0, 1.0, (n_edges, 2))
    frame = oracle.se3_oplus(np.array([0, 0, 0, 1.0, 0, 0, 0]), rng.normal(0, 0.01, 6))[None]
    i32, z = np.int32, np.zeros
    mono = synth.BAProblem(uv.astype(np.float32), pt.astype(i32), z(n_edges, i32), cam.astype(i32), z(n_edges, i32),
                           np.ones(n_edges, np.float32), points, frame, cams, z(1, i32))
    spt = np.sort(rng.choice(P - 1, n_stereo, replace=False)).astype(i32)
    xs = points[spt]
    obs = np.c_[500 * xs[:, :2] / xs[:, 2:] + [320, 240], 500 * xs[:, 0] / xs[:, 2] + 320 - 50 / xs[:, 2]]
    obs = (obs + rng.normal(0, 1.0, obs.shape)).astype(np.float32)
    stereo = synth.StereoProblem(obs, spt, z(n_stereo, i32), np.ones(n_stereo, np.float32), points, frame,
                                 np.array([500, 500, 320, 240, 50, 2.8]))
    return mono, stereo


@pytest.mark.parametrize("n_edges,n_cams,n_stereo,one_launch",
                         [(511, 1, 0, True), (512, 2, 0, True), (513, 3, 2, True), (1535, 3, 511, True),
                          (1536, 3, 512, True), (1537, 3, 513, True), (16384, 8, 0, True), (15000, 8, 1384, True),
                          (16385, 8, 0, False), (15000, 8, 1385, False), (900, 8, 40, True), (900, 9, 40, False)])
def test_single_pose_route_limits(gpu_ctx, n_edges, n_cams, n_stereo, one_launch):
    """The one-launch optimizer at the edges of its division of the edges (512
    threads, 3 mono edges each at a time) and on both sides of its limits (16384
    edges, 8 cameras), against the FP64 oracle and the general route, which the
    same problem takes when the unseen point is left free.  Tolerances as
    test_single_pose_route_vs_oracle_and_general_route."""
    mono, stereo = _one_frame(n_edges, n_cams, n_stereo, n_edges + n_cams)
    stereo = stereo if n_stereo else None
    out = []
    for last in (1, 0):
        pfix = np.ones(len(mono.points), np.int32)
        pfix[-1] = last
        lin = local_ba_linearizer(mono, stereo, pfix, ctx=gpu_ctx)
        stats, _ = lin.optimize(5)
        out.append((stats, lin.get_state()[1]))

        def again():
            lin.set_state(mono.points, mono.frames, mono.cams)
            lin.optimize(1)

        names = device_events(again, ["k_pose_optimize" if one_launch and last else "k_schur_assemble"])
        assert any("k_pose_optimize" in n for n in names) == bool(one_launch and last)
        lin.close()
    _, frs, ost, _, _ = oracle.ba_lm(mono, stereo, iterations=5, point_fixed=np.ones(len(mono.points), np.int32))
    for stats, got in out:
        assert np.abs(got[0, 4:] - frs[0, 4:]).max() < 1e-5
        assert np.abs(got[0, :4] - frs[0, :4]).max() < 1e-6
        assert abs(stats[0, 0] - ost[0, 0]) < 1e-5 * ost[0, 0]
        assert abs(stats[-1, 1] - ost[-1, 1]) < 1e-5 * ost[-1, 1]


@pytest.mark.parametrize("free,accepted", [(7723, True), (7724, False)])
def test_schur_most_free_frames(gpu_ctx, free, accepted):
    """S of 7723 free keyframes has the most entries that 31 bits count; each
    keyframe sees a point of its own and one that its neighbours see."""
    import ctypes
    from mcvslam_amd import Context
    from mcvslam_amd._native import lib
    ctx = Context(0)
    P = 2 * free
    pt = np.sort(np.r_[np.arange(P), np.arange(1, P, 2)])
    fr = np.where(np.r_[True, pt[1:] != pt[:-1]], pt // 2, np.minimum(pt // 2 + 1, free - 1))
    M = len(pt)
    lin = BALinearizer(M, P, free, 1, ctx)
    lin.set_observations(np.full((M, 2), 300.0), pt, fr, np.zeros(M), np.ones(M))
    lin.set_state(np.tile([0.1, 0.2, 5.0], (P, 1)), np.tile([0, 0, 0, 1.0, 0, 0, 0], (free, 1)),
                  [[500, 500, 320, 240, 0, 0, 0, 1.0, 0, 0, 0, 2.4]])
    lin.set_fixed(np.zeros(free))
    lin.linearize()
    assert lib().mcv_ba_schur(lin.h, ctypes.c_float(10.0)) == (0 if accepted else -1)
    ctx.synchronize()
    lin.close()
    ctx.close()
