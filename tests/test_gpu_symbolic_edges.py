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
