"""The device's symbolic analysis at the sizes where its kernels change: one word and more per
row of the pattern's bitmap, and bitmaps up to and beyond what a workgroup keeps in LDS (4096
words: 512 blocks). Every array is compared with the host analysis, whole numbers, exactly."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cams,points,constant", [(2, 3, 1), (64, 400, 0), (65, 400, 0), (66, 257, 1),
                                                  (512, 900, 0), (513, 900, 0), (514, 900, 1)])
def test_pattern_sizes_match_host(sg, cams, points, constant):
    p = sg.generate_ba(sg.BaSpec(layout=1, num_cameras=cams, num_points=points, geometric_p=0.2, seed=cams))
    order = np.random.default_rng(cams).permutation(len(p.obs_idx))
    again = np.r_[order, order[: len(order) // 10]]  # a tenth of the observations twice
    p = dataclasses.replace(p, obs_idx=p.obs_idx[again], obs_uv=p.obs_uv[again])
    v = (sg.VarBuilder()
         .add_family("cams", sg.VarFamily(sg.VarKind.Conditioned, sg.VarType.Pinhole, p.intrinsics))
         .add_family("poses", sg.VarFamily(sg.VarKind.Free, sg.VarType.Isometry3, p.poses_init,
                                           list(range(constant))))
         .add_family("points", sg.VarFamily(sg.VarKind.Marginalized, sg.VarType.Vec3, p.points_init))
         .build())
    r = sg.symbolic_check(v, p.cost_fns(1.0))
    assert r["mismatches"] == 0
    assert r["s_blocks"] >= cams - constant


@pytest.mark.parametrize("first", [0, 700_000, 1_999_500])
def test_mostly_unobserved_points(sg, first):
    """2M points of which 500 are observed, at the start, inside and at the end: the lists over the
    points have to be made in parallel where values are missing too (a serial chain there took
    48 of 63 ms)."""
    p = sg.generate_ba(sg.BaSpec(layout=0, num_cameras=10, num_points=500, obs_per_point_ring=5, seed=1))
    points = np.zeros((2_000_000, 3))
    points[:, 2] = 5.0
    points[first:first + 500] = p.points_init
    p = dataclasses.replace(p, points_init=points, obs_idx=p.obs_idx + np.array([0, 0, first]))
    runs = [sg.symbolic_check(p.variables(), p.cost_fns(1.0)) for _ in range(4)]
    assert all(r["mismatches"] == 0 for r in runs)
    device, host = (min(r[k] for r in runs) for k in ("device_ms", "host_ms"))
    print(f"first {first}: device {device:.2f} ms, host {host:.2f} ms", flush=True)
    assert device <= 2.0 * host
