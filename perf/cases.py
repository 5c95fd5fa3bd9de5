"""Performance cases: the work that programs using this package have it do, through its public entry points.

A case is a dict of plain values; "kind" says which entry point it goes through:
  window     SchurComplementBundlerGpu.solve, the drop-in call of a SLAM pipeline: one window from host buffers, packed,
             uploaded, solved and read back in the call (the pipeline has a new window every time)
  resident   SchurComplementBundlerGpu.batch + run + read: windows resident on the GPU, one solve and its results
  map        the same with one large multi-camera map (more than 40 free key frames)
  gradients  autograd.solve and its backward: gradients of a pose loss with respect to pixels and intrinsics
  inertial   IMUBundlerGpuFixedVel.solve: the visual-inertial window from host buffers
  mono       MonoSolverGpu.solve_batch: monocular windows from host buffers

Sizes are those of the repository's benchmark, presets and tests, and spread around them in draw().
"""
from __future__ import annotations

import dataclasses
import functools
import math

import numpy as np
import torch

import cuvslam_amd as ca
from cuvslam_amd import autograd, imu, imu_scene, mono

FX, FY, CX, CY = 450.0, 450.0, 376.0, 240.0
NEAR = 0.1                       # observations nearer than this to a camera are skipped
EPS = 1.1920928955078125e-07     # single-precision epsilon, the solvers' stop constant


def listed():
    return [
        # The window a tracker solves at every key frame: 7 key frames of which 3 fixed, the Student-t loss with scale
        # 0.5, 7 iterations with the early exit.
        dict(name="window_production", kind="window", scene="pinhole", key_frames=7, fixed=3, points=2000, iterations=7,
             loss="student", scale=0.5, outliers=0.02, early_exit=True),
        # The smallest call: a stereo rig's first key frames, a few hundred points, every point seen by both cameras.
        dict(name="window_small_stereo", kind="window", scene="stereo", key_frames=5, fixed=2, points=211, iterations=7,
             loss="student", scale=0.5, outliers=0.0, early_exit=True),
        # A long window from host buffers, every point seen wherever it projects (528k observations).
        dict(name="window_30kf", kind="window", scene="pinhole", key_frames=30, fixed=2, points=20000, iterations=10,
             loss="huber", scale=1.0, outliers=0.02, early_exit=False),
        # The same window resident on the GPU: offline refinement that solves it again and again.
        dict(name="resident_30kf", kind="resident", windows=1, key_frames=30, fixed=2, points=20000, iterations=10,
             loss="huber", outliers=0.02),
        # A serving or training batch of uneven windows: 5 to 40 key frames, 500 to 8000 points, up to 10% outliers.
        dict(name="batch_128_uneven", kind="resident", windows=128, key_frames=40, fixed=3, points=8000, iterations=10,
             loss="student", outliers=0.10),
        # Map refinement: an 8-camera rig, 200 key frames round a loop, 200k points, 3M observations.
        dict(name="map_200kf", kind="map", stereo_pairs=4, key_frames=200, points=200000, iterations=10,
             loss="student", outliers=0.03),
        # A smaller map of a stereo rig with odd sizes and short tracks, just past the window path's 40 free key frames.
        dict(name="map_57kf", kind="map", stereo_pairs=1, key_frames=57, points=23457, iterations=10, loss="student",
             outliers=0.0),
        # A differentiable solve: forward to convergence, refinement, and the implicit backward (180k observations).
        dict(name="gradients_20kf", kind="gradients", key_frames=20, points=9000, iterations=50, loss="student"),
        # The inertial window of a running tracker, 4-frame tracks.
        dict(name="inertial_10kf", kind="inertial", key_frames=10, fixed=1, points=800, track=4, init=False),
        # The inertial initialization: 20 key frames, 5900 points on short tracks, a strong accelerometer prior.
        dict(name="inertial_20kf_init", kind="inertial", key_frames=20, fixed=1, points=5900, track=2, init=True),
        # One monocular window, as a tracker calls it.
        dict(name="mono_window", kind="mono", windows=1, frames=8, tracks=300),
        # Monocular windows of many sequences in one call.
        dict(name="mono_batch_256", kind="mono", windows=256, frames=8, tracks=300),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["window", "window", "resident", "resident", "map", "gradients", "inertial", "mono"])
    if kind == "window":
        scene = rng.choice(["pinhole", "pinhole", "stereo"])
        loss = rng.choice(["student", "student", "huber"])
        return dict(kind=kind, scene=scene, key_frames=rng.randint(16 if loss == "huber" else 7, 40),
                    fixed=rng.randint(2, 3), points=log_int(200, 4000) if scene == "stereo" else log_int(500, 20000),
                    iterations=rng.choice([7, 10]), loss=loss, scale=rng.choice([0.5, 1.0]),
                    outliers=round(rng.uniform(0.0, 0.02 if loss == "huber" else 0.05), 3),
                    early_exit=rng.random() < 0.5)
    if kind == "resident":
        windows = rng.choice([1, log_int(2, 16), log_int(16, 128)])
        loss = "student" if windows > 1 else rng.choice(["student", "huber"])
        return dict(kind=kind, windows=windows, key_frames=rng.randint(16 if windows == 1 else 8, 40), fixed=3,
                    points=log_int(1000, 8000) if windows > 1 else log_int(1000, 20000), iterations=10, loss=loss,
                    outliers=round(rng.uniform(0.0, 0.02 if loss == "huber" else 0.10), 3))
    if kind == "map":
        pairs = rng.choice([1, 2, 4])  # short tracks (few cameras): wrong matches are found before the map is refined
        return dict(kind=kind, stereo_pairs=pairs, key_frames=log_int(44, 200), points=log_int(5000, 120000),
                    iterations=10, loss="student", outliers=0.03 if pairs == 4 else 0.0)
    if kind == "gradients":
        return dict(kind=kind, key_frames=rng.randint(6, 24), points=log_int(300, 10000), iterations=50, loss="student")
    if kind == "inertial":
        kf = rng.randint(7, 20)
        return dict(kind=kind, key_frames=kf, fixed=rng.randint(1, 2), points=log_int(200, 6000),
                    track=rng.randint(2, min(kf, 7)), init=rng.random() < 0.5)
    return dict(kind=kind, windows=log_int(1, 256), frames=rng.randint(5, 10), tracks=log_int(60, 500))


# ---- inputs -------------------------------------------------------------------------------------------------------


def _loss(case):
    return ca.LOSS_STUDENT_T if case.get("loss", "huber") == "student" else ca.LOSS_HUBER


def _landmarks(make, count, surplus, whole_tracks=False, parallax=0.75):
    """`count` landmarks of the problem that make(number of points) gives, as a SLAM front-end hands them over:
    triangulated and gated. They are seen at least four times (in every key frame with `whole_tracks`), their rays
    `parallax` degrees (root mean square) from their mean or more, and at most a tenth of their observations are much
    further than usual (five times the median) from where the initial state puts them."""
    while True:
        p = make(int(count * surplus) + 16)
        n, i, j, c = p.points.shape[0], p.point_ids, p.pose_ids, p.camera_ids
        total = lambda v=None: np.bincount(i, v, minlength=n)  # noqa: E731
        T = np.einsum("cab,kbd->kcad", p.camera_from_rig.astype(np.float64), p.rig_from_world.astype(np.float64))[j, c]
        X = p.points[i].astype(np.float64)
        q = (T[:, :3, :3] @ X[:, :, None])[:, :, 0] + T[:, :3, 3]
        off = np.abs(q[:, :2] / np.maximum(q[:, 2:], NEAR) - p.observation_xys).max(1)
        ray = X + (T[:, :3, :3].transpose(0, 2, 1) @ T[:, :3, 3:])[:, :, 0]
        ray /= np.linalg.norm(ray, axis=1, keepdims=True)
        seen = np.maximum(total(), 1)
        spread = 1.0 - np.linalg.norm(np.stack([total(ray[:, a]) for a in range(3)], 1), axis=1) / seen
        least = p.rig_from_world.shape[0] if whole_tracks else 4
        keep = ((seen >= least) & (2 * spread > math.radians(parallax) ** 2) &
                (total(off > 5 * np.median(off)) <= 0.1 * seen))
        if keep.sum() >= count:
            break
        surplus *= 1.5
    some = np.flatnonzero(keep)
    keep[:] = False
    keep[some[np.linspace(0, len(some) - 1, count).astype(int)]] = True  # spread over the scene
    o = keep[i]
    return dataclasses.replace(p, points=p.points[keep], observation_xys=p.observation_xys[o],
                               observation_infos=p.observation_infos[o], pose_ids=j[o], camera_ids=c[o],
                               point_ids=(np.cumsum(keep) - 1)[i[o]].astype(np.int32), _keep=[])


def _pinhole(case, seed, whole_tracks=False, surplus=2.0, **scene):
    truth = []

    def make(n):
        p, _, t = ca.scene.generate(seed=seed, num_points=n, num_keyframes=case["key_frames"],
                                    num_fixed_keyframes=case["fixed"], outlier_rate=case.get("outliers", 0.0),
                                    max_iterations=case["iterations"], **scene)
        p.robustifier_scale = case.get("scale", 1.0)
        truth[:] = [t]
        return p

    p = _landmarks(make, case["points"], 1.2 if case["key_frames"] >= 20 and not scene else surplus, whole_tracks)
    return p, truth[0]


def _rotation(w):
    """Rotation vectors (..., 3) to matrices (..., 3, 3)."""
    t = np.linalg.norm(w, axis=-1)[..., None, None]
    K = np.zeros(w.shape[:-1] + (3, 3))
    K[..., 0, 1], K[..., 0, 2], K[..., 1, 2] = -w[..., 2], w[..., 1], -w[..., 0]
    K -= K.swapaxes(-1, -2).copy()
    t = np.maximum(t, 1e-12)
    return np.eye(3) + np.sin(t) / t * K + (1 - np.cos(t)) / t ** 2 * K @ K


def _stereo(case, seed):
    """A two-camera rig (0.125 m baseline) moving through points 2 to 16 m away, pixel noise 0.5 px."""
    kf = case["key_frames"]

    def make(npt):
        rng = np.random.default_rng(seed)
        poses = np.tile(np.eye(4), (kf, 1, 1))  # rig_from_world
        poses[:, :3, :3] = _rotation(rng.normal(0, 0.03, (kf, 3)))
        poses[:, :3, 3] = np.stack([-0.2 * np.arange(kf), rng.normal(0, 0.02, kf), rng.normal(0, 0.02, kf)], 1)
        pts = np.stack([rng.uniform(-4, 4, npt) + 0.1 * kf, rng.uniform(-3, 3, npt), rng.uniform(2, 16, npt)], 1)
        cams = np.tile(np.eye(4), (2, 1, 1))
        cams[1, 0, 3] = -0.125
        q = np.einsum("cab,kbd,dn->kcan", cams, poses, np.concatenate([pts, np.ones((npt, 1))], 1).T)[:, :, :3]
        uv = q[:, :, :2] / np.maximum(q[:, :, 2:], 0.5)
        kid, cid, pid = np.nonzero((q[:, :, 2] > 1.0) & (np.abs(uv[:, :, 0]) < 0.9) & (np.abs(uv[:, :, 1]) < 0.6))
        xy = uv[kid, cid, :, pid] + rng.normal(0, 0.5 / FX, (len(kid), 2))
        wrong = rng.random(len(kid)) < case.get("outliers", 0.0)
        xy[wrong] = rng.uniform(-0.6, 0.6, (int(wrong.sum()), 2))
        start = poses.copy()
        free = kf - case["fixed"]  # the fixed key frames are stored last
        start[:free, :3, :3] = _rotation(rng.normal(0, 0.005, (free, 3))) @ start[:free, :3, :3]
        start[:free, :3, 3] += rng.normal(0, 0.02, (free, 3))
        return ca.BundleAdjustmentProblem(
            (pts + rng.normal(0, 0.05, pts.shape)).astype(np.float32), xy.astype(np.float32),
            np.tile(np.diag([FX * FX, FY * FY]).astype(np.float32), (len(kid), 1, 1)), pid.astype(np.int32),
            kid.astype(np.int32), cid.astype(np.int8), start.astype(np.float32), cams.astype(np.float32), 0,
            case["fixed"], case["iterations"], case.get("scale", 1.0))

    return _landmarks(make, case["points"], 1.5)


def _windows(case, seed):
    if case["windows"] == 1:
        return [_pinhole(case, seed)[0]]
    # every window has its own size and outlier rate (the same for every seed); a landmark is seen from 2 to all of the
    # key frames that it projects in
    rng = np.random.default_rng(17)
    out = []
    for w in range(case["windows"]):
        one = dict(case, key_frames=int(rng.integers(5, case["key_frames"] + 1)),
                   points=int(rng.integers(max(300, case["points"] // 16), case["points"] + 1)),
                   outliers=float(rng.uniform(0.0, case["outliers"])))
        out.append(_pinhole(one, (seed * 1000 + w) % (1 << 62), surplus=4.0 if one["key_frames"] < 9 else 1.9,
                            sample_observations=1)[0])
    return out


def _map(case, seed):
    def make(n):
        return ca.scene.loop(seed=seed, max_iterations=case["iterations"], num_keyframes=case["key_frames"],
                             num_points=n, num_stereo_pairs=case["stereo_pairs"], outlier_rate=case["outliers"])[0]

    return _landmarks(make, case["points"], 1.25 if case["stereo_pairs"] == 4 else 2.0, parallax=2.5)


def _inertial(case, seed):
    p, calib, _ = imu_scene.make_scenario(seed, (case["key_frames"], case["fixed"], case["points"], case["track"]))
    return (imu_scene.use_init_settings(p) if case["init"] else p), calib


def _mono_window(rng, frames, tracks):
    """A tracker's monocular window: the oldest three frames constrained, tracks seen from two frames or more."""
    poses = np.tile(np.eye(4), (frames, 1, 1))  # world_from_camera
    poses[:, :3, :3] = _rotation(np.radians(rng.normal(0, 1.0, (frames, 3))))
    poses[:, :3, 3] = np.stack([0.1 * np.arange(frames), 0.02 * np.sin(np.arange(frames)), np.zeros(frames)], 1)
    points = np.zeros((0, 3))
    while len(points) < tracks:
        n = 2 * tracks
        new = np.stack([rng.uniform(-4, 4, n), rng.uniform(-3, 3, n), rng.uniform(4, 15, n)], 1)
        points = np.concatenate([points, new[_in_view(poses, new)[0].sum(0) >= 2]])
    points = points[:tracks]
    seen, uv = _in_view(poses, points)
    f, t = np.nonzero(seen)
    xy = uv[f, t] + rng.normal(0, 0.5 / FX, (len(f), 2))
    start = poses.copy()
    start[3:, :3, :3] = _rotation(np.radians(rng.normal(0, 0.3, (frames - 3, 3)))) @ start[3:, :3, :3]
    start[3:, :3, 3] += rng.normal(0, 0.01, (frames - 3, 3))
    return dict(constrained=(np.arange(frames) < 3).astype(np.int32), frame_poses=start.astype(np.float32),
                points=(points + rng.normal(0, 0.05, points.shape)).astype(np.float32), obs_frame=f.astype(np.int32),
                obs_track=t.astype(np.int32), obs_xy=xy.astype(np.float32), max_iterations=30, min_residual=0.02,
                min_residual_speed=0.1)


def _in_view(poses, pts):
    q = np.einsum("fba,ftb->fta", poses[:, :3, :3], pts[None] - poses[:, None, :3, 3])
    uv = q[..., :2] / q[..., 2:]
    return (q[..., 2] > 1.0) & (np.abs(uv[..., 0]) < 0.8) & (np.abs(uv[..., 1]) < 0.5), uv


def _mono(case, seed):
    rng = np.random.default_rng(seed)
    return [_mono_window(rng, case["frames"], case["tracks"]) for _ in range(case["windows"])]


@functools.lru_cache(maxsize=None)
def _solver(loss, fixed_iterations):
    """A program keeps one solver handle for all its windows."""
    return ca.SchurComplementBundlerGpu(loss=loss, fixed_iterations=fixed_iterations)


@functools.lru_cache(maxsize=None)
def _mono_solver():
    return mono.MonoSolverGpu()


@functools.lru_cache(maxsize=None)
def _inertial_solver():
    return imu.IMUBundlerGpuFixedVel(imu_scene.calibration())


def _host_problem(case, seed):
    return _stereo(case, seed) if case["scene"] == "stereo" else _pinhole(case, seed)[0]


def _gradient_inputs(case, seed):
    p, truth = _pinhole(dict(case, fixed=2), seed, whole_tracks=True)
    uv = p.observation_xys.astype(np.float64) * [FX, FY] + [CX, CY]
    return p, uv, truth.astype(np.float64)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "window":
        return dict(kind=kind, solver=_solver(_loss(case), not case["early_exit"]), problem=_host_problem(case, seed))
    if kind in ("resident", "map"):
        problems = [_map(case, seed)] if kind == "map" else _windows(case, seed)
        return dict(kind=kind, batch=_solver(_loss(case), True).batch(problems), problems=problems)
    if kind == "gradients":
        p, uv, truth = _gradient_inputs(case, seed)
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        return dict(kind=kind, solver=_solver(_loss(case), True), template=p,
                    pixels=torch.from_numpy(uv).to(dev).requires_grad_(),
                    intrinsics=torch.tensor([FX, FY, CX, CY], dtype=torch.float64, device=dev, requires_grad=True),
                    target=torch.from_numpy(truth).to(dev))
    if kind == "inertial":
        return dict(kind=kind, solver=_inertial_solver(), problem=_inertial(case, seed)[0])
    return dict(kind=kind, solver=_mono_solver(), windows=_mono(case, seed))


def run(state):
    kind = state["kind"]
    if kind == "window":
        p = dataclasses.replace(state["problem"], _keep=[])  # solve() puts new points and key frames into it
        state["solver"].solve(p)
        return p.points, p.rig_from_world, np.array([p.initial_cost_f64, p.last_cost_f64])
    if kind in ("resident", "map"):
        state["batch"].run()
        ps = [dataclasses.replace(p, _keep=[]) for p in state["problems"]]
        state["batch"].read(ps)
        return (np.concatenate([p.points for p in ps]), np.concatenate([p.rig_from_world for p in ps]),
                np.array([[p.initial_cost_f64, p.last_cost_f64] for p in ps]))
    if kind == "gradients":
        poses, points = autograd.solve(state["pixels"], state["intrinsics"], state["template"], state["solver"])
        loss = ((poses - state["target"]) ** 2).sum()
        d_pixels, d_intrinsics = torch.autograd.grad(loss, (state["pixels"], state["intrinsics"]))
        return poses.detach(), points.detach(), d_pixels, d_intrinsics
    if kind == "inertial":
        p = dataclasses.replace(state["problem"], _keep=[])
        state["solver"].solve(p)
        return (p.points, p.w_from_imu, p.velocity, p.gyro_bias, p.acc_bias,
                np.array([p.initial_cost_f64, p.last_cost_f64]))
    out = state["solver"].solve_batch(state["windows"])
    return (np.concatenate([o["points"] for o in out]), np.concatenate([o["frame_poses"] for o in out]),
            np.stack([o["covariance"] for o in out]),
            np.array([[o["residual_initial"], o["residual"]] for o in out]))


# ---- what a pass cannot do without --------------------------------------------------------------------------------


def _visual_work(p, iterations):
    """Bytes of the problem and its result once, and the operations of each iteration: linearization, normal
    equations, Schur products of every point's pairs, factor, back-substitution and trial cost."""
    ncf = p.rig_from_world.shape[0] - p.num_fixed_key_frames
    no, npt, nc = p.num_observations, p.points.shape[0], p.rig_from_world.shape[0]
    pairs = np.unique(p.point_ids.astype(np.int64) * nc + p.pose_ids)
    q = np.bincount(pairs[pairs % nc < ncf] // nc, minlength=npt).astype(np.float64)
    n = 6.0 * ncf
    flops = 760.0 * no + 600.0 * npt + (108.0 * q * (q - 1) + 270.0 * q).sum() + n ** 3 / 3 + 2 * n * n
    return dict(bytes=33.0 * no + 24.0 * npt + 128.0 * nc, flops=float(iterations * flops))


def work(case):
    kind = case["kind"]
    if kind == "window":
        return _visual_work(_host_problem(case, 1), case["iterations"])
    if kind == "map":
        return _visual_work(_map(case, 1), case["iterations"])
    if kind == "resident":
        parts = [_visual_work(p, case["iterations"]) for p in _windows(case, 1)]
        return {k: sum(w[k] for w in parts) for k in ("bytes", "flops")}
    if kind == "gradients":
        # the forward solve, then at least one Hessian product and one preconditioner per observation and step of the
        # refinement (3 steps) and of the backward, about 20 conjugate-gradient iterations each
        p = _gradient_inputs(case, 1)[0]
        w = _visual_work(p, case["iterations"])
        no = p.num_observations
        return dict(bytes=w["bytes"] + 24.0 * no, flops=w["flops"] + 4 * 20 * 900.0 * no)
    if kind == "inertial":
        p = _inertial(case, 1)[0]
        no, npt, n = p.num_observations, p.points.shape[0], 15.0 * (case["key_frames"] - case["fixed"])
        pairs = no / 2.0
        return dict(bytes=33.0 * no + 24.0 * npt + 1500.0 * case["key_frames"],
                    flops=10 * (700.0 * no + 300.0 * npt + 108.0 * pairs * case["track"] + n ** 3 / 3))
    no = sum(len(w["obs_frame"]) for w in _mono(dict(case, windows=min(case["windows"], 16)), 1))
    no *= case["windows"] / min(case["windows"], 16)
    n = 6.0 * (case["frames"] - 3)
    return dict(bytes=16.0 * no + 24.0 * case["windows"] * case["tracks"],
                flops=8 * (900.0 * no + 108.0 * no * (case["frames"] - 3) + case["windows"] * n ** 3))


def tolerance(case):
    # Visual solves: packed in other chunk sizes (other orders of the single-precision sums) the listed windows and maps
    # move by up to 5e-7 (points) in the 2-norm and 8e-5 at the worst point, less well determined windows by up to 2e-6
    # and 4e-4. Gradients (refined in double precision) differ by up to 9e-12. The inertial and monocular solves are double
    # precision with results rounded to single precision: 1e-7, and up to 7e-7 against exact().
    kind = case["kind"]
    if kind in ("window", "resident", "map"):
        return {"rel": 1e-5, "max": 2e-3}
    if kind == "gradients":
        return {"rel": 1e-10, "max": 1e-8}
    return {"rel": 2e-6, "max": 1e-4}


# ---- 64-bit references --------------------------------------------------------------------------------------------


class _Exact:
    """The Levenberg-Marquardt solve of one visual window in plain 64-bit torch."""

    def __init__(self, p, student):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        to = lambda a, t=torch.float64: torch.as_tensor(np.ascontiguousarray(a)).to(self.dev, t)  # noqa: E731
        self.student, self.delta = student, float(p.robustifier_scale)
        self.xy = to(p.observation_xys)
        info = to(p.observation_infos)
        self.info = 0.5 * (info + info.transpose(1, 2))
        self.i, self.j, c = to(p.point_ids, torch.int64), to(p.pose_ids, torch.int64), to(p.camera_ids, torch.int64)
        cams = to(p.camera_from_rig)
        self.Rc, self.tc = cams[c, :3, :3], cams[c, :3, 3]
        self.T, self.X = to(p.rig_from_world)[:, :3], to(p.points)
        self.nf = self.T.shape[0] - p.num_fixed_key_frames
        self.np = self.X.shape[0]
        nc = self.T.shape[0]
        pair, self.pair_of = torch.unique(self.i * nc + self.j, return_inverse=True)
        self.pi, self.pj = pair // nc, pair % nc
        self.pfree = self.pj < self.nf
        # ranges of whole points whose dense blocks fit in memory
        first = torch.searchsorted(self.pi, torch.arange(self.np + 1, device=self.dev))
        step = max(64, int(6e7 / max(1, 6 * self.nf) / 3))
        self.ranges = [(a, min(a + step, self.np), int(first[a]), int(first[min(a + step, self.np)]))
                       for a in range(0, self.np, step)]

    def points_in_camera(self, T, X):
        q = (T[self.j, :, :3] @ X[self.i, :, None]).squeeze(-1) + T[self.j, :, 3]
        return q, (self.Rc @ q[..., None]).squeeze(-1) + self.tc

    def rho(self, s):
        d = self.delta
        if self.student:
            return (d + 1) * torch.log1p(s / d)
        return torch.where(s < d * d, 0.5 * s, d * torch.sqrt(torch.clamp(s, min=d * d)) - 0.5 * d * d)

    def drho(self, s):
        d = self.delta
        if self.student:
            return (d + 1) / (d + s)
        return torch.where(s < d * d, torch.full_like(s, 0.5), 0.5 * d / torch.sqrt(torch.clamp(s, min=d * d)))

    def square(self, r):
        return (r * (self.info @ r[..., None]).squeeze(-1)).sum(-1)

    def cost(self, T, X):
        _, c = self.points_in_camera(T, X)
        ok = c[:, 2] > NEAR
        z = torch.where(ok, c[:, 2], torch.ones_like(c[:, 2]))
        return torch.where(ok, self.rho(self.square(self.xy - c[:, :2] / z[:, None])), torch.zeros_like(z)).sum()

    def linearize(self, T, X):
        q, c = self.points_in_camera(T, X)
        ok = c[:, 2] > NEAR
        z = torch.where(ok, c[:, 2], torch.ones_like(c[:, 2]))
        uv = c[:, :2] / z[:, None]
        r = self.xy - uv
        A = (self.Rc[:, :2] - uv[..., None] * self.Rc[:, 2:]) / z[:, None, None]  # projection times camera rotation
        self.Jc = torch.cat([torch.cross(q[:, None].expand_as(A), A, dim=-1), A], -1)
        self.Jp = A @ T[self.j, :, :3]
        self.w = self.drho(self.square(r)) * ok
        L = self.w[:, None, None] * self.info
        LJc, LJp, Lr = L @ self.Jc, L @ self.Jp, (L @ r[..., None])
        zeros = lambda *n: torch.zeros(*n, dtype=torch.float64, device=self.dev)  # noqa: E731
        self.U = self.by_pose(self.j, self.Jc.mT @ LJc)[:self.nf]
        self.ea = self.by_pose(self.j, (self.Jc.mT @ Lr).squeeze(-1))[:self.nf]
        self.V = zeros(self.np, 3, 3).index_add_(0, self.i, self.Jp.mT @ LJp)
        self.eb = zeros(self.np, 3).index_add_(0, self.i, (self.Jp.mT @ Lr).squeeze(-1))
        self.W = zeros(self.pi.shape[0], 6, 3).index_add_(0, self.pair_of, self.Jc.mT @ LJp)
        self.W[~self.pfree] = 0

    def by_pose(self, j, v):
        """Sums of v over equal key frames j, in 256 partial sums so that few terms meet at one address."""
        n = self.T.shape[0]
        part = torch.zeros(256 * n, *v.shape[1:], dtype=torch.float64, device=self.dev)
        slot = j * 256 + torch.arange(len(j), device=self.dev) % 256
        return part.index_add_(0, slot, v).reshape(n, 256, *v.shape[1:]).sum(1)

    def inverse_points(self, lam):
        """Damped point blocks, inverted on the eigenvalues above 1e-6 of the largest (none when fewer than two are)."""
        V = self.V + lam * torch.diag_embed(torch.diagonal(self.V, dim1=1, dim2=2))
        det = torch.linalg.det(V)
        tr = torch.diagonal(V, dim1=1, dim2=2).sum(1)
        m2 = 0.5 * (tr * tr - (V * V).sum((1, 2)))
        sure = (det > 4e-6 * tr * m2) & (m2 > 0) & (tr > 0)
        out = torch.zeros_like(V)
        out[sure] = torch.linalg.inv(V[sure])
        rest = (~sure).nonzero().squeeze(-1)
        if len(rest):
            e, Q = torch.linalg.eigh(V[rest].cpu())
            keep = (e > 1e-6 * e.abs().amax(1, keepdim=True)) & (e > 0)
            keep &= keep.sum(1, keepdim=True) >= 2
            out[rest] = (Q @ torch.diag_embed(torch.where(keep, 1 / e, 0.0)) @ Q.mT).to(self.dev)
        return out

    def reduced(self, lam):
        """Factor of the damped reduced system (None when it is not positive definite)."""
        self.Vi = self.inverse_points(lam)
        n = 6 * self.nf
        U = self.U + lam * torch.diag_embed(torch.diagonal(self.U, dim1=1, dim2=2))
        S = torch.block_diag(*U) if self.nf else torch.zeros(0, 0, dtype=torch.float64, device=self.dev)
        for a, e, qa, qe in self.ranges:
            f = self.pfree[qa:qe]
            B = torch.zeros(self.nf, e - a, 6, 3, dtype=torch.float64, device=self.dev)
            B[self.pj[qa:qe][f], self.pi[qa:qe][f] - a] = self.W[qa:qe][f]
            C = (B @ self.Vi[a:e]).transpose(1, 2).reshape(n, -1)
            S = S - B.transpose(1, 2).reshape(n, -1) @ C.T
        F, bad = torch.linalg.cholesky_ex(S)
        return None if int(bad) else F

    def back(self, F, ea, eb):
        """The step (pose twists, points) of the factored system for a right-hand side."""
        t = (self.Vi @ eb[..., None])[self.pi]
        rhs = ea - self.by_pose(self.pj, (self.W @ t).squeeze(-1))[:self.nf]
        dc = torch.cholesky_solve(rhs.reshape(-1, 1), F).reshape(self.nf, 6)
        full = torch.cat([dc, torch.zeros(self.T.shape[0] - self.nf, 6, dtype=torch.float64, device=self.dev)])
        s = torch.zeros(self.np, 3, dtype=torch.float64, device=self.dev).index_add_(
            0, self.pi, (self.W.mT @ full[self.pj][..., None]).squeeze(-1))
        return full, (self.Vi @ (eb - s)[..., None]).squeeze(-1)

    def move(self, T, dc):
        """Exp(dc) T, rotations projected back onto the rotation group."""
        E = torch.zeros(T.shape[0], 4, 4, dtype=torch.float64, device=self.dev)
        w = dc[:, :3]
        E[:, 0, 1], E[:, 0, 2], E[:, 1, 2] = -w[:, 2], w[:, 1], -w[:, 0]
        E = E - E.mT
        E[:, :3, 3] = dc[:, 3:]
        E = torch.linalg.matrix_exp(E)[:, :3]
        R, t = E[:, :, :3] @ T[:, :, :3], (E[:, :, :3] @ T[:, :, 3:]) + E[:, :, 3:]
        Us, _, Vs = torch.linalg.svd(R.cpu())
        return torch.cat([torch.cat([(Us @ Vs).to(self.dev), t], -1)[:self.nf], T[self.nf:]])

    def solve(self, iterations, early_exit):
        T, X, lam = self.T, self.X, 1e-3
        cost = first = float(self.cost(T, X))
        fresh = False
        for _ in range(iterations):
            if not fresh:
                self.linearize(T, X)
                fresh = True
            F = self.reduced(lam)
            if F is None:
                lam *= 5
                continue
            dc, dp = self.back(F, self.ea, self.eb)
            Tn, Xn = self.move(T, dc), X + dp
            trial = float(self.cost(Tn, Xn))
            step = (self.Jc @ dc[self.j][..., None] + self.Jp @ dp[self.i][..., None]).squeeze(-1)
            pred = float((self.w * self.square(step)).sum() + 2 * lam * (
                (dc[:self.nf] ** 2 * torch.diagonal(self.U, dim1=1, dim2=2)).sum() +
                (dp ** 2 * torch.diagonal(self.V, dim1=1, dim2=2)).sum())) / cost
            if cost < first * EPS or (early_exit and pred < math.sqrt(EPS) and
                                      max(float(dc.abs().max()), float(dp.abs().max())) < math.sqrt(EPS)):
                break
            ratio = (1 - trial / cost) / pred
            if ratio > 0.25:
                T, X, cost, fresh = Tn, Xn, trial, False
                lam *= 0.125 if ratio > 0.75 else 1.0
            else:
                lam *= 5
        return T, X, first, cost

    def gradients(self, T, X, uv, target):
        """Newton steps to the stationary point, then the implicit gradient of sum (T - target)^2 with respect to the
        pixels and (fx, fy, cx, cy), all derivatives of the cost by automatic differentiation."""
        nc, nf = T.shape[0], self.nf
        uv = torch.from_numpy(uv).to(self.dev)
        K = torch.tensor([FX, FY, CX, CY], dtype=torch.float64, device=self.dev)
        d = self.delta

        def F(x, T, X, uv, K):
            tw, dx = x[:6 * nf].reshape(nf, 6), x[6 * nf:].reshape(-1, 3)
            w, v = tw[:, :3], tw[:, 3:]
            R, t = T[:nf, :, :3], T[:nf, :, 3]
            cross = lambda a, b: torch.cross(a, b, dim=-1)  # noqa: E731
            Rw = lambda B: torch.cross(w[:, :, None].expand_as(B), B, dim=1)  # noqa: E731
            Rn = R + Rw(R) + 0.5 * Rw(Rw(R))  # Exp to second order: exact for the Hessian at x = 0
            tn = t + cross(w, t) + v + 0.5 * cross(w, cross(w, t) + v)
            Ts = torch.cat([torch.cat([Rn, tn[..., None]], -1), T[nf:]])
            q, c = self.points_in_camera(Ts, X + dx)
            r = (uv - K[2:]) / K[:2] - c[:, :2] / c[:, 2:]
            s = ((r * K[:2]) ** 2).sum(-1)
            return ((d + 1) * torch.log1p(s / d)).sum()

        x0 = torch.zeros(6 * nf + 3 * self.np, dtype=torch.float64, device=self.dev)

        def derivative(T, X, inputs=()):
            x = x0.clone().requires_grad_()
            g, = torch.autograd.grad(F(x, T, X, *(inputs or (uv, K))), x, create_graph=True)
            return x, g

        def newton(rhs, T, X, x, g):
            """H^-1 rhs by conjugate gradients, preconditioned with the factored Gauss-Newton system."""
            self.linearize(T, X)
            fac = self.reduced(0.0)

            def precondition(r):
                dc, dp = self.back(fac, r[:6 * nf].reshape(nf, 6), r[6 * nf:].reshape(-1, 3))
                return 0.5 * torch.cat([dc[:nf].reshape(-1), dp.reshape(-1)])

            y, r = torch.zeros_like(rhs), rhs.clone()
            z = precondition(r)
            s, rz, norm = z, r @ z, rhs.norm()
            for _ in range(200):
                h, = torch.autograd.grad(g, x, s, retain_graph=True)
                curve = s @ h
                if not float(curve) > 0:
                    break
                y, r = y + rz / curve * s, r - rz / curve * h
                if float(r.norm()) < 1e-13 * float(norm):
                    break
                z = precondition(r)
                rz, old = r @ z, rz
                s = z + rz / old * s
            return y

        for k in range(10):
            x, g = derivative(T, X)
            if k < 4:
                self.linearize(T, X)
                dc, dp = self.back(self.reduced(0.0), self.ea, self.eb)
            else:
                a = newton(-g.detach(), T, X, x, g)
                dc = torch.cat([a[:6 * nf].reshape(nf, 6), x0.new_zeros(nc - nf, 6)])
                dp = a[6 * nf:].reshape(-1, 3)
            T, X = self.move(T, dc), X + dp
        x, g = derivative(T, X)
        D = 2 * (T - torch.from_numpy(target[:, :3]).to(self.dev))[:nf]
        A = D[..., :3] @ T[:nf, :, :3].mT + D[..., 3:] @ T[:nf, :, 3:].mT
        gw = torch.stack([A[:, 2, 1] - A[:, 1, 2], A[:, 0, 2] - A[:, 2, 0], A[:, 1, 0] - A[:, 0, 1]], 1)
        a = newton(torch.cat([torch.cat([gw, D[..., 3]], 1).reshape(-1), x0[6 * nf:]]), T, X, x, g)
        uvg, Kg = uv.clone().requires_grad_(), K.clone().requires_grad_()
        _, g = derivative(T, X, (uvg, Kg))
        duv, dK = torch.autograd.grad(g @ a, (uvg, Kg))
        return T, X, -duv, -dK


def _square(T):
    """(n, 3, 4) poses as (n, 4, 4)."""
    out = torch.eye(4, dtype=torch.float64).repeat(T.shape[0], 1, 1)
    out[:, :3] = T.cpu()
    return out


class _ExactMono:
    """The monocular solve of one window in plain 64-bit numpy: Huber loss on each track's own information, damping
    times or over 10, one frame pose camera_from_world per frame."""

    def __init__(self, w):
        T = w["frame_poses"].astype(np.float64)
        self.R = T[:, :3, :3].transpose(0, 2, 1).copy()
        self.t = -np.einsum("fab,fb->fa", self.R, T[:, :3, 3])
        self.b = w["points"].astype(np.float64)
        self.f, self.k, self.xy = w["obs_frame"], w["obs_track"], w["obs_xy"].astype(np.float64)
        self.free = np.cumsum(w["constrained"] == 0) - 1
        self.free[w["constrained"] != 0] = -1
        self.w, self.skip = w, np.zeros(len(self.b), bool)
        self.info, self.err = np.tile(np.eye(2), (len(self.b), 1, 1)), np.zeros_like(self.xy)

    def camera(self, R, t, b):
        return np.einsum("oab,ob->oa", R[self.f], b[self.k]) + t[self.f]

    def behind(self):
        self.skip[self.k[~(self.camera(self.R, self.t, self.b)[:, 2] > NEAR)]] = True

    def squares(self, err):
        return np.einsum("oa,oab,ob->o", err, self.info[self.k], err)

    def residual(self, R, t, b):
        q = self.camera(R, t, b)
        self.err = np.where(self.skip[self.k][:, None], self.err, self.xy - q[:, :2] / q[:, 2:])
        s = self.squares(self.err)[~self.skip[self.k]]
        return np.where(s < 0.25, 0.5 * s, 0.5 * np.sqrt(s) - 0.125).mean() if len(s) else math.inf

    def information(self):
        floor = float(np.float32(1e-5))
        n = np.bincount(self.k, minlength=len(self.b)).astype(float)
        mean = lambda v: np.bincount(self.k, v, minlength=len(self.b)) / n  # noqa: E731
        ex, ey = self.err.T
        mx, my, mxy = mean(ex), mean(ey), mean(ex * ey)
        vx, vy = mean((ex - mx[self.k]) ** 2), mean((ey - my[self.k]) ** 2)
        for i in np.nonzero(~self.skip)[0]:
            c = np.diag([max(vx[i], floor), max(vy[i], floor)])
            if n[i] > 3:
                p00, p11, p01 = max(c[0, 0], c[1, 1]), min(c[0, 0], c[1, 1]), mxy[i] - mx[i] * my[i]
                if not abs(c[1, 1]) > abs(c[0, 0]):
                    p00, p11 = c[0, 0], c[1, 1]
                low = p01 / p00
                e0, e1 = max(p00, floor), max(p11 - low * p01, floor)
                c = np.array([[e0, low * e0], [low * e0, low * low * e0 + e1]])
            det = c[0, 0] * c[1, 1] - c[0, 1] * c[1, 0]
            self.info[i] = (np.array([[c[1, 1], -c[0, 1]], [-c[1, 0], c[0, 0]]]) / det if abs(det) > EPS
                            else np.diag([1 / c[0, 0], 1 / c[1, 1]]))

    def system(self):
        use, fr = ~self.skip[self.k], self.free[self.f]
        q = self.camera(self.R, self.t, self.b)
        iz = 1 / q[:, 2]
        x, y, o = q[:, 0] * iz, q[:, 1] * iz, np.zeros(len(iz))
        U_, _, V_ = np.linalg.svd(self.R)
        Rn = (U_ @ V_)[self.f]
        B = np.stack([Rn[:, 0] - Rn[:, 2] * x[:, None], Rn[:, 1] - Rn[:, 2] * y[:, None]], 1) * iz[:, None, None]
        A = -np.stack([x * y, -x * x - 1, y, -iz, o, x * iz, y * y + 1, -x * y, -x, o, -iz, y * iz], 1)
        A = A.reshape(-1, 2, 6)
        s = self.squares_weight
        L = (s * use)[:, None, None] * self.info[self.k]
        n, m = 6 * (self.free.max() + 1), len(self.b)
        self.A6, self.V, self.eB = np.zeros((n // 6, 6, 6)), np.zeros((m, 3, 3)), np.zeros((m, 3))
        self.eA, mv = np.zeros((n // 6, 6)), fr >= 0
        Le = np.einsum("oab,ob->oa", L, self.err)
        np.add.at(self.V, self.k, B.transpose(0, 2, 1) @ L @ B)
        np.add.at(self.eB, self.k, np.einsum("oab,oa->ob", B, Le))
        np.add.at(self.A6, fr[mv], (A.transpose(0, 2, 1) @ L @ A)[mv])
        np.add.at(self.eA, fr[mv], np.einsum("oab,oa->ob", A, Le)[mv])
        self.Wd = np.zeros((n // 6, m, 6, 3))
        self.Wd[fr[mv], self.k[mv]] = (A.transpose(0, 2, 1) @ L @ B)[mv]

    def step(self, lam):
        V = self.V * (1 + lam * np.eye(3))
        det = np.linalg.det(V)
        self.skip |= ~(np.abs(det) > 1 / max(1e6, lam ** 3))
        X = np.zeros_like(V)
        ok = ~self.skip
        X[ok] = np.linalg.inv(V[ok])
        W = self.Wd * ok[None, :, None, None]
        n, Y = 6 * len(W), W @ X
        flat = lambda M: M.transpose(0, 2, 1, 3).reshape(n, -1)  # noqa: E731
        S = -flat(Y) @ flat(W).T
        for j in range(len(W)):
            S[6 * j:6 * j + 6, 6 * j:6 * j + 6] += self.A6[j] * (1 + lam * np.eye(6))
        self.last = S[n - 6:, n - 6:].copy()
        self.last[np.diag_indices(6)] /= 1 + lam
        e = np.linalg.eigvalsh(0.5 * (S + S.T))
        if not np.all(np.abs(e) > n * EPS * np.abs(e).max()):
            return None
        dc = np.linalg.solve(S, (self.eA.reshape(-1) - flat(Y) @ self.eB.reshape(-1))).reshape(-1, 6)
        db = np.einsum("tab,tb->ta", X, self.eB - np.einsum("jtab,ja->tb", W, dc))
        R, t = self.R.copy(), self.t.copy()
        for f in np.nonzero(self.free >= 0)[0]:
            xi = np.zeros((4, 4))
            w, v = dc[self.free[f], :3], dc[self.free[f], 3:]
            xi[:3, :3], xi[:3, 3] = [[0, -w[2], w[1]], [w[2], 0, -w[0]], [-w[1], w[0], 0]], v
            E = torch.linalg.matrix_exp(torch.from_numpy(xi)).numpy()
            R[f], t[f] = E[:3, :3] @ R[f], E[:3, :3] @ t[f] + E[:3, 3]
        return R, t, self.b + db * ok[:, None]

    def weights(self):
        s = self.squares(self.err)
        self.squares_weight = np.where(s < 0.25, 0.5, 0.25 / np.sqrt(np.maximum(s, 0.25)))

    def covariance(self):
        e, Q = np.linalg.eigh(0.5 * (self.last + self.last.T))
        keep = np.abs(e) > 6 * EPS * np.abs(e).max()
        return (Q[:, keep] / e[keep]) @ Q[:, keep].T

    def solve(self):
        w, lam, count, fresh = self.w, float(np.float32(0.001)), self.w["max_iterations"], True
        self.behind()
        self.residual(self.R, self.t, self.b)
        self.information()
        self.weights()
        res = old = first = self.residual(self.R, self.t, self.b)
        cov = np.zeros((6, 6))
        speed, least = (float(np.float32(w[k])) for k in ("min_residual_speed", "min_residual"))
        while least <= res and count >= 0 and lam <= 1e7:
            if fresh:
                self.system()
            new = self.step(lam)
            res = self.residual(*new) if new is not None else 2 * res
            delta = abs(res - old)
            if res > old:
                lam, fresh = lam * 10, False
            else:
                lam, old, fresh = lam / 10, res, True
                moved = ~self.skip
                self.R, self.t = new[0], new[1]
                self.b[moved] = new[2][moved]
                self.skip[:] = False
                self.behind()
                self.information()
                self.weights()
                cov = self.covariance()
            if speed * res > delta:
                break
            count -= 1
        if lam > 1e7 or count < 0:
            cov = self.covariance()
        T = np.tile(np.eye(4), (len(self.R), 1, 1))
        T[:, :3, :3] = self.R.transpose(0, 2, 1)
        T[:, :3, 3] = -np.einsum("fba,fb->fa", self.R, self.t)
        return self.b, T, cov, np.array([first, old])


def exact(case, seed):
    kind = case["kind"]
    if kind == "mono":
        return tuple(np.concatenate(x) if n < 2 else np.stack(x)
                     for n, x in enumerate(zip(*[_ExactMono(w).solve() for w in _mono(case, seed)])))
    if kind == "inertial":
        return None  # 64-bit throughout, to 1e-14 of its own definition: tolerance() holds it
    if kind == "gradients":
        p, uv, truth = _gradient_inputs(case, seed)
        e = _Exact(p, case["loss"] == "student")
        T, X, _, _ = e.solve(case["iterations"], False)
        T, X, duv, dK = e.gradients(T, X, uv, truth)
        return _square(T), X, duv, dK
    make = {"window": _host_problem, "map": _map, "resident": _windows}[kind]
    ps = make(case, seed) if kind == "resident" else [make(case, seed)]
    out = [_Exact(p, case["loss"] == "student").solve(p.max_iterations, case.get("early_exit", False)) for p in ps]
    costs = np.array([o[2:] for o in out], np.float64)
    return (torch.cat([o[1].cpu() for o in out]), torch.cat([_square(o[0]) for o in out]),
            costs[0] if kind == "window" else costs)
