"""The forward solve of the supernodal factor at its edges: one pivot block, exactly one and
two panels of 48 columns, one block more, and nodes with more rows below a panel than the
workgroup takes in one pass (448). Blocks of the damped Hessian's inverse against numpy's
dense inverse.

Bound: a solve with a stable factorization in the scaling D = diag(H), Hs = D^-1/2 H D^-1/2,
is off by at most c n eps cond(Hs) |Hs^-1| (Higham, Accuracy and Stability, 10.1; the scaling
drops out of the factorization). c = 4 covers the product with the points' blocks."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cams,points", [(2, 40), (9, 60), (10, 60), (17, 80), (18, 80), (95, 500)])
def test_inverse_blocks_match_dense_inverse(sg, orc, cams, points):
    p = sg.generate_ba(sg.BaSpec(layout=0, num_cameras=cams, num_points=points, obs_per_point_ring=0, min_obs=2,
                                 max_obs=min(8, cams), seed=cams))
    opt = sg.Optimizer(p.variables(), p.cost_fns(1.0),
                       sg.OptParams(num_iterations=3, initial_lm_damping=1.0, skip_final_hessian=True))
    while opt.step().termination is None:
        pass
    H, _ = orc.linearize_dense(orc.ba_families(p, opt.members("poses"), opt.members("points")), orc.ba_costs(p),
                               opt.lm_damping())
    s = 1.0 / np.sqrt(np.diag(H))
    Hs = H * s[:, None] * s
    Hinv = np.linalg.inv(Hs)
    w = np.linalg.eigvalsh(Hs)
    bound = 4 * len(H) * np.finfo(float).eps * (w[-1] / w[0]) / w[0]
    nfree = 6 * (cams - 1)
    index = {"poses": lambda m: slice(6 * (m - 1), 6 * m), "points": lambda m: slice(nfree + 3 * m, nfree + 3 * m + 3)}
    worst = 0.0
    for rf, rm, cf, cm in [("poses", 1, "poses", cams - 1), ("poses", cams - 1, "poses", cams - 1),
                           ("poses", 1 + cams // 2 if cams > 2 else 1, "points", 7),
                           ("points", points - 1, "points", 3)]:
        r, c = index[rf](rm), index[cf](cm)
        blk = opt.inverse_block(rf, rm, cf, cm) / s[r][:, None] / s[c]
        worst = max(worst, float(np.max(np.abs(blk - Hinv[r, c]))))
    print(f"{cams} cameras: error {worst:.2g}, bound {bound:.2g}, 1 / smallest eigenvalue {1 / w[0]:.2g}")
    assert worst <= bound
    assert worst <= 1e-6 / w[0]
    opt.close()
