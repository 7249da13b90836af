"""BA linearization on the GPU (FP32, compensated residual) against the
FP64 oracle of EdgeSE3XYZ2Camera (include/OptimizeTypes.hpp:70-117)."""
import numpy as np
import pytest

import oracle
from mcvslam_amd import BALinearizer, synth

pytestmark = pytest.mark.gpu

from ba_check import TOL, check_against_oracle, rel_rows


def test_ba_150k(gpu_ctx):
    prob = synth.ba_problem(seed=30, n_kf=10, n_points=20000, target_obs=150000)
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize()
    check_against_oracle(prob, b.results())
    assert (b.results()[2] < 1).sum() > 0.03 * len(prob.obs_pt)   # outliers hit the Huber branch


def test_ba_perturbed_state(gpu_ctx):
    """State with full FP64 precision (not float-representable)."""
    prob = synth.ba_problem(seed=31, n_kf=6, n_points=3000, target_obs=30000, perturb=0.01)
    prob.frames[:, 4:] += np.random.default_rng(1).normal(0, 1e-3, (len(prob.frames), 3))
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize()
    check_against_oracle(prob, b.results())


def test_ba_reference_huber_deltas(gpu_ctx):
    """LEFT edges use sqrt(5.99), WIDE sqrt(7.815) (src/BAoptimizer.cpp:62,105)."""
    prob = synth.ba_problem(seed=32, n_kf=4, n_points=2000, target_obs=20000)
    prob.cams[:, 11] = [np.float32(np.sqrt(5.99)), np.float32(np.sqrt(7.815)), np.float32(np.sqrt(7.815))]
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize()
    check_against_oracle(prob, b.results())


def test_ba_plain_equals_batched(gpu_ctx):
    """One launch per (frame, camera) group gives the same bits as the
    all-edges launch (the pair table comes from LDS in one, from global
    memory in the other)."""
    prob = synth.ba_problem(seed=34, n_kf=5, n_points=4000, target_obs=30000)
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize()
    batched = b.read()
    b.linearize_plain()
    np.testing.assert_array_equal(b.read(), batched)


def test_ba_every_launch_variant(gpu_ctx):
    """Every launch shape (workgroup size, grid cap, observations in flight,
    streaming stores) writes the same bits.  Before each variant the planes
    are overwritten from a shifted state, so a variant that skips
    observations fails."""
    prob = synth.ba_problem(seed=36, n_kf=5, n_points=4000, target_obs=30011)
    assert len(prob.obs_pt) % 256 != 0
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.set_variant(0)
    b.linearize()
    ref = b.read()
    check_against_oracle(prob, b.results())
    shifted = prob.points + 0.25
    for v in range(1, BALinearizer.N_VARIANTS):
        b.set_variant(0)
        b.set_state(shifted, prob.frames, prob.cams)
        b.linearize()
        assert not np.array_equal(b.read(0, 1), ref[:1])
        b.set_state(prob.points, prob.frames, prob.cams)
        b.set_variant(v)
        b.linearize()
        np.testing.assert_array_equal(b.read(), ref, err_msg=f"variant {v}")
    rep = b.autotune(reps=2)
    assert rep.count("k_ba_linearize") == BALinearizer.N_VARIANTS + 1
    np.testing.assert_array_equal(b.read(), ref)
    with pytest.raises(Exception):
        b.set_variant(BALinearizer.N_VARIANTS)


def test_ba_many_pairs(gpu_ctx):
    """More (frame, camera) pairs than the LDS copy holds (70 x 3 = 210)."""
    prob = synth.ba_problem(seed=35, n_kf=70, n_points=6000, target_obs=40000)
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize()
    check_against_oracle(prob, b.results())


def test_ba_residual_only(gpu_ctx):
    prob = synth.ba_problem(seed=33, n_kf=3, n_points=1000, target_obs=8000)
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize(residual_only=True)
    pl = b.read(0, 4)
    re, rchi2, rw, _, _ = oracle.ba_linearize(prob)
    assert rel_rows(np.stack([pl[0], pl[1]], 1), re, 1e-9).max() < TOL


@pytest.mark.parametrize("lam", [1e2, 1e4])
def test_schur_vs_fp64(gpu_ctx, lam):
    """FP32 reduced camera system against the FP64 oracle (dense elimination
    is pinned in test_oracle_match_ba.py); the FP64 host Cholesky solves both
    to the same pose step.  lambda is in the range g2o's LM starts from
    (tau = 1e-5 times the largest diagonal entry, optimization_algorithm_
    levenberg.cpp); lambda = 0 leaves single-observation points singular."""
    prob = synth.ba_problem(seed=35, n_kf=8, n_points=6000, target_obs=60000)
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize()
    S, bs = b.schur(lam)
    e, chi2, w, Jp, Jx = oracle.ba_linearize(prob)
    r = oracle.ba_schur(e, w, Jp, Jx, prob.obs_pt, prob.obs_frame, prob.obs_isig, len(prob.points),
                        len(prob.frames), prob.frame_fixed, lam)
    assert S.shape == r["S"].shape
    assert np.linalg.norm(S - r["S"]) / np.linalg.norm(r["S"]) < 1e-5
    assert np.linalg.norm(bs - r["bs"]) / np.linalg.norm(r["bs"]) < 1e-4
    if True:
        x = b.solve_llt(S, bs)
        xr = np.linalg.solve(r["S"], r["bs"])
        assert np.linalg.norm(x - xr) / np.linalg.norm(xr) < 1e-3
    b.close()


def _without_damping(seed):
    """Points of one edge, whose H_ll has rank 2, among points whose H_ll has
    a condition number below 300; per point (frames, J_pose, J_point, W, e)."""
    prob = synth.ba_problem(seed=seed, n_kf=5, n_points=700, target_obs=7000)
    e, _, w, Jp, Jx = oracle.ba_linearize(prob)
    W = w * prob.obs_isig
    Hll = np.zeros((len(prob.points), 3, 3))
    np.add.at(Hll, prob.obs_pt, W[:, None, None] * np.einsum("mri,mrj->mij", Jx, Jx))
    good = np.linalg.cond(Hll) < 300
    first = np.r_[True, prob.obs_pt[1:] != prob.obs_pt[:-1]]
    keep = good[prob.obs_pt] | first
    for k in ("obs_uv", "obs_pt", "obs_frame", "obs_cam", "obs_level", "obs_isig"):
        setattr(prob, k, getattr(prob, k)[keep])
    n = np.bincount(prob.obs_pt, minlength=len(prob.points))
    assert (n == 1).sum() > 100 and (n > 1).sum() > 100
    return prob, n


def test_schur_without_damping(gpu_ctx):
    """lambda = 0, the default: points of one edge contribute what the
    pseudo-inverse of their H_ll does, and keep S and b_schur finite.  Bound:
    16 roundings of 2^-24 at a condition number of 300, of the sums of the
    magnitudes (a pivot left out lies under 2^-23 of its diagonal and what
    remains of its column within 16 roundings, so it would add less)."""
    prob, n = _without_damping(36)
    lin = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    lin.linearize()
    S, bs = lin.schur()
    e, _, w, Jp, Jx = oracle.ba_linearize(prob)
    free = np.nonzero(prob.frame_fixed == 0)[0]
    col = {f: 6 * k for k, f in enumerate(free)}
    m = 6 * len(free)
    want, mag = (np.zeros((m, m + 1)) for _ in range(2))
    for p in np.unique(prob.obs_pt):
        i = np.nonzero(prob.obs_pt == p)[0]
        W = (w[i] * prob.obs_isig[i]).repeat(2)[:, None]
        A = np.zeros((2 * len(i), m))
        for k, j in enumerate(i):
            if prob.obs_frame[j] in col:
                c = col[prob.obs_frame[j]]
                A[2 * k:2 * k + 2, c:c + 6] = Jp[j]
        B, r = Jx[i].reshape(-1, 3), e[i].reshape(-1, 1)
        AB = (W * A).T @ B
        rest = np.linalg.pinv((W * B).T @ B, rcond=1e-9) @ np.c_[AB.T, -(W * B).T @ r]
        want += np.c_[(W * A).T @ A, -(W * A).T @ r] - AB @ rest
        mag += np.c_[np.abs(W * A).T @ np.abs(A), np.abs(W * A).T @ np.abs(r)] + np.abs(AB) @ np.abs(rest)
    assert np.isfinite(S).all() and np.isfinite(bs).all()
    tol = 16 * 2.0 ** -24 * 300
    assert np.linalg.norm(S - want[:, :m]) < tol * np.linalg.norm(mag[:, :m])
    assert np.linalg.norm(bs - want[:, m]) < tol * np.linalg.norm(mag[:, m])
    # undamped steps: points without parallax no longer stop the optimizer
    stats, _ = lin.optimize(3, tau=0.0)
    assert np.isfinite(stats).all() and stats[-1, 1] < stats[0, 0]
    assert all(np.isfinite(x).all() for x in lin.get_state())
    lin.close()


def test_stereo_edge_vs_oracle(gpu_ctx):
    """EdgeStereoSE3ProjectXYZ on the GPU against the FP64 oracle: residual,
    chi2, Huber weight and the 3x6 / 3x3 Jacobians within 1e-5."""
    sp = synth.stereo_problem(seed=54, n_kf=8, n_points=6000, target_obs=20000)
    base = synth.ba_problem(seed=54, n_kf=8, n_points=6000, target_obs=60000, outlier_frac=0.05)
    b = BALinearizer.from_problem(base, ctx=gpu_ctx)
    b.set_stereo(sp.obs, sp.obs_pt, sp.obs_frame, sp.obs_isig, sp.cam)
    b.linearize_stereo()
    e, chi2, w, Jp, Jx = b.stereo_results()
    re, rchi2, rw, rJp, rJx = oracle.ba_stereo_linearize(sp.obs, sp.obs_pt, sp.obs_frame, sp.obs_isig, sp.points,
                                                         sp.frames, sp.cam)
    assert rel_rows(e, re, 1e-9).max() < TOL
    assert (np.abs(chi2 - rchi2) / np.maximum(rchi2, 1e-12)).max() < TOL
    d2 = sp.cam[5] ** 2
    ok = np.abs(rchi2 - d2) > 1e-6 * d2
    assert (np.abs(w - rw)[ok] / rw[ok]).max() < TOL
    assert (w < 1).sum() > 0
    for r in range(3):
        assert rel_rows(Jp[:, r], rJp[:, r]).max() < TOL, f"J_pose row {r}"
        assert rel_rows(Jx[:, r], rJx[:, r]).max() < TOL, f"J_point row {r}"


def test_outlier_flags(gpu_ctx):
    """chi2 >= threshold on the GPU's chi2 planes, and the oracle's flags
    wherever chi2 is not within 1e-5 of the threshold."""
    prob = synth.ba_problem(seed=55, n_kf=5, n_points=3000, target_obs=20000)
    b = BALinearizer.from_problem(prob, ctx=gpu_ctx)
    b.linearize()
    chi2 = b.results()[1]
    thr = float(np.float32(5.991))
    fm, _ = b.outliers(thr, 7.815)
    np.testing.assert_array_equal(fm, (chi2 >= np.float32(thr)).astype(np.uint8))
    _, rchi2, _, _, _ = oracle.ba_linearize(prob)
    want = oracle.ba_outliers(rchi2, thr)
    far = np.abs(rchi2 - thr) > 1e-5 * thr
    np.testing.assert_array_equal(fm[far], want[far])
    assert 0 < fm.sum() < len(fm)
