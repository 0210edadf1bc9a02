"""Coarse levels with variable coefficients (banded plans) fused into one workgroup: the V-cycle
gives the solution and defect history of the separate launches bit for bit, in every precision of
the cycle, with all of the boundary filtered (every computed row has its 3^dim neighbours) or one
face of it (clipped rows are computed too), and for step counts of either parity."""
import numpy as np
import pytest

from tests.helpers import q1_levels

pytestmark = pytest.mark.gpu


def lognormal_levels(feat, dim, lf, lc, one_face):
    if dim == 3:
        levels = feat.diffusion3d_levels(lf, lc, 515, 1.5, 10.0)
    else:
        levels = [dict(q) for q in q1_levels(feat, 2, lf, lc)]
        coef = feat.lognormal_cells(516, 4 ** lf, 1.5)
        for k, q in zip(range(lf, lc - 1, -1), levels):
            q["val"] = feat.q1_diffusion(k, lf, coef)
    if one_face:
        for k, q in zip(range(lf, lc - 1, -1), levels):
            q["filt"] = np.ascontiguousarray(q["filt"][q["filt"] % (2 ** k + 1) == 0])
    return levels


@pytest.mark.parametrize("precision", ["f64", "f32", "f16"])
@pytest.mark.parametrize("dim,lf,lc,first,nu,one_face", [
    (3, 4, 1, 1, (4, 4), False),     # 729 and 125 rows over 27
    (3, 5, 2, 2, (1, 3), True),      # 729 rows over 125
    (2, 6, 2, 2, (3, 2), True),      # 289 and 81 rows over 25
])
def test_banded_coarse_fusion_bitwise(feat, torch_gpu, dim, lf, lc, first, nu, one_face, precision):
    print(f"banded coarse fusion {precision} dim={dim} levels {lf}..{lc} V{nu} one face {one_face}", flush=True)
    torch = torch_gpu
    levels = lognormal_levels(feat, dim, lf, lc, one_face)
    n = levels[0]["n"]
    b = feat.rhs_random(31, n, -1.0, 1.0)
    b[levels[0]["filt"].astype(np.int64)] = 0.0
    bd = torch.from_numpy(b).cuda()
    out = []
    for fusion in (True, False):
        s = feat.MgPcg(feat.mgpcg_cfg(nu_pre=nu[0], nu_post=nu[1], omega_jac=0.5, omega_rich=1.0, coarse="direct",
                                      tol_rel=1e-8, max_iter=300, graphs=False, coarse_fusion=fusion,
                                      precision=precision), levels=levels)
        assert s.coarse_fusion_level() == (first if fusion else 0)
        x = torch.zeros(n, dtype=torch.float64, device="cuda")
        r = s.solve(x, bd)
        torch.cuda.synchronize()
        s.close()
        assert r["status"] == "success"
        out.append((r, x.cpu().numpy()))
    (r1, x1), (r0, x0) = out
    assert r1["iters"] == r0["iters"]
    assert np.array_equal(r1["hist"].view(np.uint64), r0["hist"].view(np.uint64))
    assert np.array_equal(x1.view(np.uint64), x0.view(np.uint64))
