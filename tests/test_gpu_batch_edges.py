"""Batched windows at the edges of the window kernel's tiling: reduced systems of one 6-column
panel, one and several 12-column panels with and without a remainder, the largest (31
cameras), points seen by every camera (many segments of shared points per camera pair),
repeated observations of a point by one camera, and a camera without observations (six
zero pivots).  Each window against the FP64 oracle run on it alone, with the bars of the
batch tests in FP64 (1e-9 on the cost, 1e-7 on the variables).  With FP32 Schur products the
cost's bar is 1e-5: a product's rounding (6e-8 relative) enters S, whose free scale leaves these
small windows' condition number above 1e2 after the damping falls; two summation orders of
the same products differ by up to 6e-6 here after ten iterations."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _window(sg, nc, npt, obs, seed, repeats=0, idle=False):
    p = sg.generate_ba(sg.BaSpec(layout=0, num_cameras=nc, num_points=npt, obs_per_point_ring=obs, seed=seed))
    rng = np.random.default_rng(seed)
    if repeats:  # the same (camera, point) again, once and twice, with its own pixel
        k = np.r_[rng.choice(p.num_obs, repeats, replace=False)]
        k = np.r_[k, k[: repeats // 2]]
        p = dataclasses.replace(p, obs_idx=np.vstack([p.obs_idx, p.obs_idx[k]]),
                                obs_uv=np.vstack([p.obs_uv, p.obs_uv[k] + rng.normal(0, 0.3, (k.size, 2))]))
    if idle:
        p = dataclasses.replace(p, poses_init=np.vstack([p.poses_init, p.poses_init[1:2]]),
                                poses_gt=np.vstack([p.poses_gt, p.poses_gt[1:2]]))
    return p


def _cases(sg):
    return [_window(sg, 2, 12, 2, 1), _window(sg, 3, 20, 3, 2), _window(sg, 4, 30, 3, 3), _window(sg, 6, 9, 6, 4),
            _window(sg, 7, 513, 7, 5), _window(sg, 12, 100, 5, 6), _window(sg, 18, 130, 18, 7),
            _window(sg, 31, 300, 4, 8), _window(sg, 5, 60, 3, 9, repeats=20), _window(sg, 9, 80, 4, 10, repeats=40),
            _window(sg, 6, 50, 4, 11, idle=True), _window(sg, 30, 40, 30, 12, repeats=10)]


@pytest.mark.parametrize("mode,mixed", [("run", False), ("run_persistent", False), ("run", True)])
def test_window_edges_match_oracle(sg, orc, mode, mixed):
    ws = _cases(sg)
    iters = 10
    b = sg.Batch(ws, sg.OptParams(num_iterations=iters, initial_lm_damping=1.0,
                                  precision=sg.Precision.Mixed if mixed else sg.Precision.F64))
    getattr(b, mode)(iters)
    res = b.results()
    for p, w in enumerate(ws):
        sol, vars_, _ = orc.optimize_nlls(orc.ba_families(w), orc.ba_costs(w),
                                          orc.default_params(num_iterations=iters, initial_lm_damping=1.0))
        rel = abs(res["final_cost"][p] - sol["final_cost"]) / sol["final_cost"]
        assert rel <= (1e-5 if mixed else 1e-9), (p, rel)
        if mixed:
            continue
        assert res["steps"][p] == sol["num_steps"] and res["termination"][p] == sol["termination"], p
        sl = b.window_slice(p)
        assert np.max(np.abs(res["poses"][sl["poses"]] - vars_["poses"])) < 1e-7, p
        assert np.max(np.abs(res["points"][sl["points"]] - vars_["points"])) < 1e-7, p
    b.close()


def test_small_and_large_batches_are_filled_alike(sg):
    """Up to 1 MiB of host values go to the device in one copy, more array by array: a window of 60 kB
    alone and 32 of it give the same runs."""
    w = _window(sg, 9, 400, 6, 13)
    params = sg.OptParams(num_iterations=8, initial_lm_damping=1.0)
    results = []
    for n in (1, 32):
        b = sg.Batch([w] * n, params)
        b.run(8)
        results.append((b.results(), [b.window_slice(p) for p in range(n)]))
        b.close()
    one, many = results
    for p, sl in enumerate(many[1]):
        assert abs(many[0]["final_cost"][p] / one[0]["final_cost"][0] - 1.0) <= 1e-9, p
        for name in ("poses", "points"):
            assert np.max(np.abs(many[0][name][sl[name]] - one[0][name])) < 1e-7, (p, name)
