"""What a user of this framework has it do, as cases that can be timed and compared.

Four calls make up the framework's use:

- ``solve``: ``optimize_nlls`` on a problem in host memory, as a program that has one bundle
  adjustment to do calls it (upload, symbolic analysis, LM iterations, variables back);
- ``iterate``: a kept ``Optimizer`` advanced by a few LM iterations, then its variables read,
  as a program that watches or steers a long run does (tolerances off, as in the benchmark);
- ``batch``: a kept ``Batch`` of small windows restarted, run and read;
- ``covariance``: the final linearization of a kept, adjusted ``Optimizer`` and blocks of its
  inverse.

Sizes are the repository's workloads (10-, 500- and 2,000-camera problems, the 10- and
120-camera EUCM rings, the windows of 5-30 cameras) and the sizes between them in its tests.
"""
from __future__ import annotations

import dataclasses
import math
import sys
from pathlib import Path

import numpy as np

ROOT = Path(__file__).resolve().parent.parent
sys.path.insert(0, str(ROOT / "sophus-rs_amd"))

import sophus_opt_gpu as sg  # noqa: E402

# ---- the cases ------------------------------------------------------------------------------

_SOLVE = {"call": "solve", "layout": "walk", "track": 0.1, "solver": "block", "mixed": False, "huber": True,
          "intrinsics": "fixed", "factors": "none", "iterations": 20}


def _case(name, **kw):
    return {"name": name, **_SOLVE, **kw}


def listed():
    return [
        # the smallest problem in the repository, with the solver its benchmark names: launches,
        # allocations and the analysis count, not arithmetic
        _case("ring10", layout="ring", cameras=10, points=200, track=5, solver="sparse"),
        # the reference's own bundle adjustment benchmark: an EUCM camera calibrated on the way
        _case("calibrate10", layout="eucm", cameras=10, points=500, huber=False, intrinsics="free"),
        # the same with the scale held by an equality constraint (odd sizes)
        _case("scale31", layout="eucm", cameras=31, points=2003, huber=False, intrinsics="free", factors="scale",
              iterations=10),
        # a local map with odometry between consecutive poses, FP32 assembly
        _case("odometry60", cameras=60, points=3000, track=0.15, mixed=True, factors="odometry", iterations=10),
        # many cameras on the same points: the EUCM ring at scale, about 50 observations a point
        _case("calibrate120", layout="eucm", cameras=120, points=12000, huber=False, intrinsics="free"),
        # one whole reconstruction of ordinary size, direct solver
        _case("walk500", cameras=500, points=100_000),
        # the same size with conjugate gradients at the default tolerance
        _case("walk499_pcg", cameras=499, points=60_001, solver="pcg", iterations=6),
        # FP32 assembly, learned preconditioner and a forcing sequence: the fast inexact path
        _case("walk1000_learned", cameras=1000, points=200_000, track=0.135, solver="learned", mixed=True,
              iterations=25),
        # the benchmark's largest problem (about 6M observations), a long run watched as it goes
        _case("walk2000", call="iterate", cameras=2000, points=800_000, track=0.135, iterations=5),
        # a live system's windows, all at once in one launch
        {"name": "windows24", "call": "batch", "windows": 24, "mode": "persistent", "mixed": False, "iterations": 20},
        # a backlog of windows, one launch per iteration, FP32 assembly
        {"name": "windows1000", "call": "batch", "windows": 1000, "mode": "launches", "mixed": True,
         "iterations": 10},
        # marginal covariances after an adjustment with pose priors
        _case("covariance150", call="covariance", cameras=150, points=8000, factors="priors", iterations=5),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ring", "eucm", "eucm", "walk", "walk", "walk", "iterate", "batch", "batch", "covariance"])
    if kind == "batch":
        return {"call": "batch", "windows": _between(rng, 16, 1000), "mode": rng.choice(["persistent", "launches"]),
                "mixed": rng.random() < 0.5, "iterations": rng.randint(5, 20)}
    if kind == "iterate":
        return {**_SOLVE, "call": "iterate", "cameras": _between(rng, 1000, 2000),
                "points": _between(rng, 200_000, 800_000), "track": rng.uniform(0.135, 0.2),
                "mixed": rng.random() < 0.25, "iterations": rng.randint(2, 5)}
    if kind == "ring":
        return {**_SOLVE, "layout": "ring", "cameras": _between(rng, 5, 60), "points": _between(rng, 100, 5000),
                "track": rng.randint(3, 5), "solver": rng.choice(["block", "sparse"]), "iterations": 20}
    if kind == "eucm":
        intr = rng.choice(["fixed", "free", "free"])
        return {**_SOLVE, "layout": "eucm", "cameras": _between(rng, 8, 120), "points": _between(rng, 300, 12000),
                "huber": False, "intrinsics": intr, "factors": "scale" if intr == "free" and rng.random() < 0.3
                else "none", "iterations": rng.randint(8, 20)}
    if kind == "covariance":
        return {**_SOLVE, "call": "covariance", "cameras": _between(rng, 20, 400), "points": _between(rng, 1000, 40_000),
                "track": rng.uniform(0.1, 0.2), "factors": "priors", "iterations": rng.randint(2, 5)}
    solver = rng.choice(["block", "block", "sparse", "pcg", "learned"])
    case = {**_SOLVE, "cameras": _between(rng, 30, 1000), "track": rng.uniform(0.1, 0.2), "solver": solver,
            "mixed": solver == "learned" or (solver != "pcg" and rng.random() < 0.4),
            "iterations": rng.randint(3, 6) if solver == "pcg" else rng.randint(5, 20),
            "factors": rng.choice(["none", "none", "odometry"])}
    return {**case, "points": max(_between(rng, 1000, 200_000), 20 * case["cameras"])}


# ---- inputs and calls -----------------------------------------------------------------------


def _eucm_problem(cameras, points, seed):
    """The EUCM ring with exactly `points` points: the generator drops the few that fewer than two
    cameras see, so it is asked for some more and the first ones are kept."""
    p = sg.generate_ba_eucm(cameras, points + points // 50 + 10, seed=seed)
    keep = p.obs_idx[:, 2] < points
    p.points_gt, p.points_init = p.points_gt[:points].copy(), p.points_init[:points].copy()
    p.obs_idx, p.obs_uv = p.obs_idx[keep], p.obs_uv[keep]
    return p


def _problem(case, seed):
    if case["layout"] == "eucm":
        return _eucm_problem(case["cameras"], case["points"], seed)
    if case["layout"] == "ring":
        return sg.generate_ba(sg.BaSpec(layout=0, num_cameras=case["cameras"], num_points=case["points"],
                                        obs_per_point_ring=int(case["track"]), seed=seed))
    return sg.generate_ba(sg.BaSpec(layout=1, num_cameras=case["cameras"], num_points=case["points"],
                                    geometric_p=case["track"], seed=seed))


def _const_poses(case):
    """Members of the pose family held constant (priors fix the gauge by themselves)."""
    if case["factors"] == "priors":
        return []
    return [0, 1] if case["layout"] == "eucm" and case["factors"] != "scale" else [0]


def _prior_members(case):
    return np.arange(0, case["cameras"], 10)


_PRIOR_PRECISION = 1e4 * np.eye(6)


def _window_specs(case, seed):
    """The repository's windows by number: their sizes are the case's, their contents the seed's."""
    return [dataclasses.replace(sg.window_spec(i), seed=seed * 1_000_003 + i) for i in range(case["windows"])]


def _odometry(p):
    """Consecutive poses and their true relative poses."""
    n = p.poses_gt.shape[0]
    pairs = np.stack([np.arange(n - 1), np.arange(1, n)], axis=1)
    return pairs, _se3_mul(_se3_inverse(p.poses_gt[:-1]), p.poses_gt[1:])


def _describe(case, p):
    """Variables, cost functions and constraints of a problem, as a user's program builds them."""
    huber = sg.RobustKernel.huber(1.0) if case["huber"] else None
    names = ["cams", "poses", "points"]
    if case["layout"] == "eucm":
        free = case["intrinsics"] == "free"
        intr = p.intrinsics_init if free else p.intrinsics_gt
        cams = sg.VarFamily(sg.VarKind.Free if free else sg.VarKind.Conditioned, sg.VarType.Eucm, intr)
        costs = [sg.CostFn.eucm_reprojection(names, p.obs_idx, p.obs_uv, huber)]
    else:
        cams = sg.VarFamily(sg.VarKind.Conditioned, sg.VarType.Pinhole, p.intrinsics)
        costs = [sg.CostFn.pinhole_reprojection(names, p.obs_idx, p.obs_uv, huber)]
    variables = (sg.VarBuilder()
                 .add_family("cams", cams)
                 .add_family("poses", sg.VarFamily(sg.VarKind.Free, sg.VarType.Isometry3, p.poses_init,
                                                   _const_poses(case)))
                 .add_family("points", sg.VarFamily(sg.VarKind.Marginalized, sg.VarType.Vec3, p.points_init))
                 .build())
    eqs = []
    if case["factors"] == "odometry":
        pairs, meas = _odometry(p)
        costs.append(sg.CostFn.pose_graph3(["poses", "poses"], pairs, meas, sg.RobustKernel.huber(0.5)))
    elif case["factors"] == "priors":
        m = _prior_members(case)
        costs.append(sg.CostFn.isometry3_prior(["poses"], m, p.poses_gt[m], _PRIOR_PRECISION))
    elif case["factors"] == "scale":
        eqs.append(sg.EqConstraintFn.translation_norm("poses", [1], [np.linalg.norm(p.poses_gt[1, 4:])]))
    return variables, costs, eqs


_SOLVERS = {"block": sg.Solver.SchurBlockSparseLdlt, "sparse": sg.Solver.SchurSparseLdlt,
            "pcg": sg.Solver.SchurPcgJacobi, "learned": sg.Solver.SchurPcgLearned}


def _params(case):
    p = sg.OptParams(num_iterations=case["iterations"], initial_lm_damping=1.0,
                     precision=sg.Precision.Mixed if case["mixed"] else sg.Precision.F64)
    if case["call"] == "batch":
        return p
    p.solver = _SOLVERS[case["solver"]]
    if case["solver"] == "pcg":
        p.pcg_max_iterations = 3000
    elif case["solver"] == "learned":
        p.precond_weights = np.fromfile(ROOT / "sophus-rs_amd" / "precond_weights.f32", dtype="<f4")
        p.pcg_max_iterations, p.pcg_forcing = 3000, 0.1
    if case["call"] == "iterate":
        p.num_iterations = p.max_consecutive_rejects = 1 << 40
        p.function_tolerance = p.gradient_tolerance = p.parameter_tolerance = 0.0
    return p


def prepare(case, seed):
    if case["call"] == "batch":
        windows = [sg.generate_ba(s) for s in _window_specs(case, seed)]
        return {"case": case, "batch": sg.Batch(windows, _params(case), huber_delta=1.0)}
    variables, costs, eqs = _describe(case, _problem(case, seed))
    state = {"case": case, "variables": variables, "costs": costs, "eqs": eqs, "params": _params(case)}
    if case["call"] in ("iterate", "covariance"):
        state["optimizer"] = sg.Optimizer(variables, costs, state["params"], eqs)
    if case["call"] == "covariance":
        while state["optimizer"].step().termination is None:
            pass
    return state


def _queries(case):
    """Pose marginals, a pair's cross block, pose-point and point-point blocks."""
    i, j, k = case["cameras"] // 2, case["cameras"] - 1, case["points"] // 3
    return [("poses", i, "poses", i), ("poses", i, "poses", j), ("poses", j, "points", k), ("points", k, "points", k)]


def run(state):
    case = state["case"]
    if case["call"] == "batch":
        b = state["batch"]
        b.reset()
        (b.run_persistent if case["mode"] == "persistent" else b.run)(case["iterations"])
        r = b.results()
        return {"poses": r["poses"], "points": r["points"], "cost": r["final_cost"]}
    if case["call"] == "covariance":
        o = state["optimizer"]
        s = o.build_solution()
        out = {"poses": s.variables.get_members("poses"), "points": s.variables.get_members("points"),
               "cost": s.final_cost}
        for n, q in enumerate(_queries(case)):
            out["block%d" % n] = o.inverse_block(*q)
        return out
    if case["call"] == "iterate":
        o = state["optimizer"]
        for _ in range(case["iterations"]):
            o.step()
        return {"poses": o.members("poses"), "points": o.members("points"), "cost": o.merit()}
    s = sg.optimize_nlls(state["variables"], state["costs"], state["params"], state["eqs"])
    out = {"poses": s.variables.get_members("poses"), "points": s.variables.get_members("points"),
           "cost": s.final_cost}
    if case["intrinsics"] == "free":
        out["intrinsics"] = s.variables.get_members("cams")
    return out


# ---- work and tolerance ---------------------------------------------------------------------


def _tracks(case):
    """(mean observations, mean observation pairs) of a point."""
    if case["layout"] == "ring":
        k = int(case["track"])
        return k, k * (k - 1) / 2
    if case["layout"] == "eucm":
        k = case["cameras"] * (0.42 if case["cameras"] >= 20 else 1.0)  # the part of the ring that sees a point
        return k, k * (k - 1) / 2
    n = p = 0.0  # geometric lengths, clipped to [2, 30]
    q = case["track"]
    for k in range(1, 1000):
        w, c = q * (1 - q) ** (k - 1), min(max(k, 2), 30)
        n, p = n + w * c, p + w * c * (c - 1) / 2
    return n, p


def work(case):
    """Inputs and outputs once (each LM iteration reads the observations and the points once
    more); the arithmetic of the Schur complement: about 400 operations an observation, 200 a
    pair of a point's observations, and a band factorization of the camera system."""
    if case["call"] == "batch":
        w, its = case["windows"], case["iterations"]  # 17.5 cameras, 1,050 points, 5 observations a point
        n, pts, cams = 5 * 1050 * w, 1050 * w, 17.5 * w
        return {"bytes": 2 * (56 * cams + 24 * pts) + 24 * n,
                "flops": its * (400 * n + 200 * 2 * n + w * 105**3 / 3)}
    its, pts, cams = case["iterations"], case["points"], case["cameras"]
    k, pairs = _tracks(case)
    band = 6 * min(cams, 45 if case["layout"] == "walk" else cams)
    factor = 6 * cams * band * band / (1 if band < 6 * cams else 3)
    step = pts * (400 * k + 200 * pairs) + factor
    if case["call"] == "covariance":
        return {"bytes": 24 * pts * k + 24 * pts + 56 * cams, "flops": step}
    if case["call"] == "iterate":
        return {"bytes": its * (24 * pts * k + 48 * pts + 112 * cams), "flops": its * step}
    return {"bytes": 40 * pts * k + its * (24 * pts * k + 48 * pts + 112 * cams), "flops": its * step}


def tolerance(case):
    """About four times what the same problems show with their points and cameras renumbered (the
    sums and the elimination in another order).  Rings and windows are well conditioned: 1e-12 in
    FP64 (a window at a decision's boundary, or in FP32, 1e-6).  The walks' camera systems are not: 3e-8
    on ordinary seeds, 5e-5 where a point lies on a camera plane; with FP32 assembly 2e-5 to 2e-4,
    with the inexact path's loose tolerance 4e-3."""
    if case["call"] == "batch":
        return {"rel": 1e-5, "max": 1e-3}
    if case["layout"] != "walk":
        return {"rel": 1e-8}
    if case["call"] == "covariance":
        return {"rel": 1e-6}
    return {"rel": 1.5e-2 if case["solver"] == "learned" else 1e-3 if case["mixed"] else 2e-4}


# ---- the same in 64 bits, from the formulas -------------------------------------------------
# Levenberg-Marquardt with a dense Schur complement in numpy: the reference's rules for the
# damping, the Huber weighting (the gradient only) and the terminations.


def _matrix(q):
    r, x, y, z = q[:, 0], q[:, 1], q[:, 2], q[:, 3]
    return np.stack([1 - 2 * (y * y + z * z), 2 * (x * y - r * z), 2 * (x * z + r * y),
                     2 * (x * y + r * z), 1 - 2 * (x * x + z * z), 2 * (y * z - r * x),
                     2 * (x * z - r * y), 2 * (y * z + r * x), 1 - 2 * (x * x + y * y)], axis=1).reshape(-1, 3, 3)


def _hat(w):
    o = np.zeros(len(w))
    return np.stack([o, -w[:, 2], w[:, 1], w[:, 2], o, -w[:, 0], -w[:, 1], w[:, 0], o], axis=1).reshape(-1, 3, 3)


def _quat_mul(a, b):
    re = a[:, 0] * b[:, 0] - np.sum(a[:, 1:] * b[:, 1:], axis=1)
    im = a[:, :1] * b[:, 1:] + b[:, :1] * a[:, 1:] + np.cross(a[:, 1:], b[:, 1:])
    return np.column_stack([re, im])


def _rotate(q, v):
    return np.einsum("nij,nj->ni", _matrix(q), v)


def _se3_mul(a, b):
    return np.column_stack([_quat_mul(a[:, :4], b[:, :4]), _rotate(a[:, :4], b[:, 4:]) + a[:, 4:]])


def _se3_inverse(a):
    q = a[:, :4] * np.array([1.0, -1, -1, -1])
    return np.column_stack([q, -_rotate(q, a[:, 4:])])


def _series(m, first):
    """Sum of m^k / (k + first)!"""
    term = np.broadcast_to(np.eye(m.shape[-1]) / math.factorial(first), m.shape).copy()
    out = term.copy()
    for k in range(1, 40):
        term = term @ m / (k + first)
        out += term
    return out


def _se3_exp(t):
    th = np.linalg.norm(t[:, :3], axis=1, keepdims=True)
    q = np.column_stack([np.cos(th / 2), 0.5 * np.sinc(th / (2 * np.pi)) * t[:, :3]])
    return np.column_stack([q, np.einsum("nij,nj->ni", _series(_hat(t[:, :3]), 1), t[:, 3:])])


def _se3_log(a):
    q = np.where(a[:, :1] < 0, -a[:, :4], a[:, :4])
    n = np.linalg.norm(q[:, 1:], axis=1, keepdims=True)
    w = q[:, 1:] * np.where(n > 1e-12, 2 * np.arctan2(n, q[:, :1]) / np.maximum(n, 1e-300), 2.0)
    u = np.linalg.solve(_series(_hat(w), 1), a[:, 4:, None])[:, :, 0]
    return np.column_stack([w, u])


def _log_jacobian(r):
    """d log(exp(x) exp(r)) / dx at x = 0."""
    ad = np.zeros((len(r), 6, 6))
    ad[:, :3, :3] = ad[:, 3:, 3:] = _hat(r[:, :3])
    ad[:, 3:, :3] = _hat(r[:, 3:])
    return np.linalg.inv(_series(ad, 1))


def _adjoint(a):
    out = np.zeros((len(a), 6, 6))
    out[:, :3, :3] = out[:, 3:, 3:] = _matrix(a[:, :4])
    out[:, 3:, :3] = _hat(a[:, 4:]) @ out[:, :3, :3]
    return out


def _pixel(intr, xc):
    """Pinhole (4 values) or EUCM (6) projection; holds for complex arguments."""
    x, y = xc[:, 0] / xc[:, 2], xc[:, 1] / xc[:, 2]
    n = 1.0
    if len(intr) == 6:
        n = intr[4] * np.sqrt(intr[5] * (x * x + y * y) + 1.0) + (1.0 - intr[4])
    return np.stack([intr[0] * x / n + intr[2], intr[1] * y / n + intr[3]], axis=1)


def _weight(r, delta, norm=None):
    if delta is None:
        return np.ones(len(r))
    n = np.linalg.norm(r, axis=1) if norm is None else norm
    rho = np.where(n <= delta, n * n, 2 * delta * n - delta * delta)
    return np.where(n > 0, np.sqrt(rho) / np.maximum(n, 1e-300), 0.0)


class _Exact:
    def __init__(self, case, p):
        self.case, self.p = case, p
        self.cam, self.pt, self.uv = p.obs_idx[:, 1], p.obs_idx[:, 2], p.obs_uv
        free = case.get("intrinsics") == "free"
        eucm = case.get("layout") == "eucm"
        self.delta = 1.0 if case.get("huber", True) else None
        self.state = [p.poses_init, p.points_init,
                      (p.intrinsics_gt if eucm and not free else p.intrinsics_init if free else p.intrinsics)[0]]
        const = _const_poses(case) if case["call"] != "batch" else [0]
        n = len(p.poses_init)
        self.block = np.full(n, -1)
        self.block[np.setdiff1d(np.arange(n), const)] = np.arange(n - len(const))
        self.nb = n - len(const)
        self.dim = 6 * self.nb + (6 if free else 0)
        self.free = free
        self.factors = case.get("factors", "none")
        self.lam = 0.0

    def camera_points(self, s):
        R = np.transpose(_matrix(s[0][:, :4]), (0, 2, 1))
        return R, np.einsum("nij,nj->ni", R[self.cam], s[1][self.pt] - s[0][self.cam, 4:])

    def pose_terms(self, s):
        """(members, residuals, Jacobians per member, weight matrix, robust weight) of the pose factors."""
        if self.factors == "odometry":
            pairs, meas = _odometry(self.p)
            mi = _se3_inverse(s[0][pairs[:, 0]])
            r = _se3_log(_se3_mul(_se3_mul(mi, s[0][pairs[:, 1]]), _se3_inverse(meas)))
            jn = _log_jacobian(r) @ _adjoint(mi)
            return pairs, r, [-jn, jn], np.eye(6), _weight(r, 0.5)
        if self.factors == "priors":
            m = _prior_members(self.case)
            r = _se3_log(_se3_mul(s[0][m], _se3_inverse(self.p.poses_gt[m])))
            return m[:, None], r, [_log_jacobian(r)], _PRIOR_PRECISION, np.ones(len(r))
        return None

    def merit(self, s):
        _, xc = self.camera_points(s)
        r = self.uv - _pixel(s[2], xc)
        f = np.sum((_weight(r, self.delta)[:, None] * r) ** 2)
        t = self.pose_terms(s)
        if t is not None:
            rw = t[4][:, None] * t[1]
            f += np.sum(rw * (rw @ t[3]))
        return float(f)

    def linearize(self, s, nu):
        """S, its right-hand side, H_fm, H_mm^-1, the two gradients."""
        h, nb, npt = 1e-30, self.nb, len(s[1])
        R, xc = self.camera_points(s)
        r = self.uv - _pixel(s[2], xc)
        rw = _weight(r, self.delta)[:, None] * r
        D = np.stack([_pixel(s[2], xc + 1j * h * np.eye(3)[k]).imag / h for k in range(3)], axis=2)
        A = D @ R[self.cam]
        Hll = np.zeros((npt, 3, 3))
        np.add.at(Hll, self.pt, np.transpose(A, (0, 2, 1)) @ A)
        Hll += nu * np.bincount(self.pt, minlength=npt)[:, None, None] * np.eye(3)
        gl = np.zeros((npt, 3))
        np.add.at(gl, self.pt, np.einsum("nij,ni->nj", A, rw))
        Hff = np.zeros((self.dim, self.dim))
        Hfm = np.zeros((self.dim, 3 * npt))
        gf = np.zeros(self.dim)
        blk = self.block[self.cam]
        use = blk >= 0
        J = A @ np.concatenate([-_hat(s[1][self.pt]), np.broadcast_to(np.eye(3), (len(A), 3, 3))], axis=2)
        diag, grad = np.zeros((nb, 6, 6)), np.zeros((nb, 6))
        np.add.at(diag, blk[use], np.transpose(J[use], (0, 2, 1)) @ J[use])
        np.add.at(grad, blk[use], -np.einsum("nij,ni->nj", J[use], rw[use]))
        diag += nu * np.bincount(blk[use], minlength=nb)[:, None, None] * np.eye(6)
        rows, cols = 6 * blk[use][:, None] + np.arange(6), 3 * self.pt[use][:, None] + np.arange(3)
        Hfm[rows[:, :, None], cols[:, None, :]] = -np.transpose(J[use], (0, 2, 1)) @ A[use]
        if self.free:
            E = -np.stack([_pixel(s[2] + 1j * h * np.eye(6)[k], xc).imag / h for k in range(6)], axis=2)
            c = 6 * nb
            Hff[c:, c:] = np.einsum("nij,nik->jk", E, E) + nu * len(E) * np.eye(6)
            gf[c:] = -np.einsum("nij,ni->j", E, rw)
            W = np.zeros((npt, 6, 3))
            np.add.at(W, self.pt, -np.transpose(E, (0, 2, 1)) @ A)
            Hfm[c:] = np.transpose(W, (1, 0, 2)).reshape(6, -1)
            C = np.zeros((nb, 6, 6))
            np.add.at(C, blk[use], np.transpose(J[use], (0, 2, 1)) @ E[use])
            Hff[:c, c:] = C.reshape(-1, 6)
            Hff[c:, :c] = C.reshape(-1, 6).T
        for b in range(nb):
            Hff[6 * b:6 * b + 6, 6 * b:6 * b + 6] += diag[b]
        gf[:6 * nb] += grad.reshape(-1)
        t = self.pose_terms(s)
        if t is not None:
            members, pr, jac, W, w = t
            for n, ms in enumerate(members):
                for a, m in enumerate(ms):
                    i = 6 * self.block[m]
                    if i < 0:
                        continue
                    gf[i:i + 6] -= jac[a][n].T @ W @ (w[n] * pr[n])
                    Hff[i:i + 6, i:i + 6] += nu * np.eye(6)
                    for b, m2 in enumerate(ms):
                        j = 6 * self.block[m2]
                        if j >= 0:
                            Hff[i:i + 6, j:j + 6] += jac[a][n].T @ W @ jac[b][n]
        Hi = np.linalg.inv(Hll)
        B = np.einsum("fpi,pij->fpj", Hfm.reshape(self.dim, npt, 3), Hi).reshape(self.dim, -1)
        return Hff - B @ Hfm.T, gf - B @ gl.reshape(-1), Hfm, Hi, gf, gl

    def advance(self, iterations):
        """The LM iterations; self.state and the final merit."""
        s, nu, merit, rejects = self.state, 1.0, self.merit(self.state), 0
        for _ in range(iterations):
            S, rhs, Hfm, Hi, gf, gl = self.linearize(s, nu)
            extra = [0.0, 0.0, 0.0]
            lam = self.lam
            if self.factors == "scale":
                t = s[0][1, 4:]
                g = np.zeros(self.dim)
                i = 6 * self.block[1] + 3
                g[i:i + 3] = t / np.linalg.norm(t)
                c = np.linalg.norm(t) - np.linalg.norm(self.p.poses_gt[1, 4:])
                gf, rhs = gf + lam * g, rhs + lam * g
                u, y = np.linalg.solve(S, np.stack([rhs, g], axis=1)).T
                d = (g @ u + c) / (g @ y)
                dx, lam, extra = u - d * y, lam - d, [d * d, -c * d, abs(d)]
            else:
                if np.max(np.abs(gf)) < 1e-14:
                    break
                dx = np.linalg.solve(S, rhs)
            dl = np.einsum("nij,nj->ni", Hi, gl - (Hfm.T @ dx).reshape(-1, 3))
            poses = s[0].copy()
            on = self.block >= 0
            poses[on] = _se3_mul(_se3_exp(dx[:6 * self.nb].reshape(-1, 6)), s[0][on])
            new = [poses, s[1] + dl, s[2] + dx[6 * self.nb:] if self.free else s[2]]
            f = self.merit(new)
            big = max(np.max(np.abs(dx)), np.max(np.abs(dl)), extra[2])
            pred = nu * (dx @ dx + np.sum(dl * dl) + extra[0]) + dx @ gf + np.sum(dl * gl) + extra[1]
            rho = (merit - f) / pred
            if big < 1e-12:
                if f < merit:
                    s, merit, self.lam = new, f, lam
                break
            if rho > 0 and f < merit:
                nu *= max(1.0 / 3.0, 1.0 - (2.0 * rho - 1.0) ** 3)
                done = (merit - f) / abs(merit) < 1e-10
                s, merit, self.lam, rejects = new, f, lam, 0
                if done:
                    break
            else:
                nu, rejects = 2.0 * nu, rejects + 1
                if rejects >= 20:
                    break
        self.state = s
        return merit

    def inverse_block(self, query):
        S, _, Hfm, Hi, _, _ = self.linearize(self.state, 0.0)
        if self.inverse is None:
            self.inverse = np.linalg.inv(S)
        parts = []
        for family, m in (query[:2], query[2:]):
            if family == "poses":
                e = np.zeros((self.dim, 6))
                e[6 * self.block[m]:6 * self.block[m] + 6] = np.eye(6)
                parts.append((e, False))
            else:
                parts.append((-Hfm[:, 3 * m:3 * m + 3] @ Hi[m], True))
        out = parts[0][0].T @ self.inverse @ parts[1][0]
        return out + Hi[query[1]] if parts[0][1] and query[:2] == query[2:] else out

    inverse = None


def exact(case, seed):
    if case["call"] == "batch":
        if case["windows"] * case["iterations"] > 500:
            return None
        done = []
        for spec in _window_specs(case, seed):
            e = _Exact(case, sg.generate_ba(spec))
            f = e.advance(case["iterations"])
            done.append((e.state[0], e.state[1], f))
        return {"poses": np.concatenate([d[0] for d in done]), "points": np.concatenate([d[1] for d in done]),
                "cost": np.array([d[2] for d in done])}
    # the fast inexact path has no exact steps; the dense coupling has to fit and take seconds
    if case["solver"] == "learned" or 18 * case["cameras"] * case["points"] * case["iterations"] > 2e8:
        return None
    e = _Exact(case, _problem(case, seed))
    f = e.advance(case["iterations"])
    out = {"poses": e.state[0], "points": e.state[1], "cost": f}
    if case["call"] == "covariance":
        for n, q in enumerate(_queries(case)):
            out["block%d" % n] = e.inverse_block(q)
    elif e.free:
        out["intrinsics"] = e.state[2][None]
    return out
