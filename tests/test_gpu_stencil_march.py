"""Diagonal plans of structured grids whose interior rows are all the same (the march over planes):
the rows equal the entry-order dictionary plan's bit for bit at grid sizes around the 62 positions
a wave covers and the planes a lane takes, with no filter, with the boundary filtered, and with
some boundary and interior rows filtered; a grid with one odd interior row keeps the code words.
3D grids below 97 nodes a side march with the descriptor's grid_closed only (a hint: the results are
those of the code words whether the boundary is filtered or not)."""
import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def grid_csr(dim, n1, odd_row=False):
    """3^dim-point stencil, every interior row alike; clipped rows with values of their own."""
    rng = np.random.default_rng(dim)
    w = rng.uniform(-1.0, 1.0, 3 ** dim)
    n = n1 ** dim
    pos = np.stack(np.meshgrid(*[np.arange(n1)] * dim, indexing="ij"), -1).reshape(n, dim)
    cols, vals, ins = [], [], []
    edge = ((pos == 0) | (pos == n1 - 1)).any(1)
    for t, o in enumerate(itertools.product((-1, 0, 1), repeat=dim)):
        q = pos + np.array(o)
        ins.append(((q >= 0) & (q < n1)).all(1))
        cols.append((q * n1 ** np.arange(dim - 1, -1, -1)).sum(1))
        vals.append(np.where(edge, 0.5 * w[t], w[t]))
    ins = np.stack(ins, 1)
    rp = np.concatenate([[0], np.cumsum(ins.sum(1))]).astype(np.int64)
    val = np.stack(vals, 1)[ins]
    if odd_row:
        val[rp[np.flatnonzero(~edge)[-1]]] = 7.0
    return val, np.stack(cols, 1)[ins].astype(np.int64), rp, edge


@pytest.mark.parametrize("dim,n1", [(2, 3), (2, 9), (2, 61), (2, 62), (2, 63), (2, 64), (2, 249), (2, 1100), (3, 3), (3, 4),
                                    (3, 7), (3, 8), (3, 16), (3, 33), (3, 64), (3, 65), (3, 96), (3, 97)])
def test_march_bitwise(feat, handle, torch_gpu, dim, n1):
    print(f"stencil march dim={dim} n1={n1}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    P = feat.ptr
    val, col, rp, edge = grid_csr(dim, n1)
    n = n1 ** dim
    dev = [torch.from_numpy(a).cuda() for a in (val, col, rp)]
    rng = np.random.default_rng(n1)
    some = edge & (rng.random(n) < 0.5) | (rng.random(n) < 0.1)
    keep, ws = feat.reduce_ws(torch, "cuda")
    for fp in ("f64", "f32"):
        dt = torch.float64 if fp == "f64" else torch.float32
        x, rhs, inv = (torch.from_numpy(rng.standard_normal(n)).cuda().to(dt) for _ in range(3))
        plans = [feat.SellPlan(handle, *dev, n, n, fp=fp), feat.SellPlan(handle, *dev, n, n, fp=fp, diag=False),
                 feat.SellPlan(handle, *dev, n, n, fp=fp)]
        plans[0].m.grid_closed = 1
        # plans whose empty slots exceed a quarter of the entries keep the entry-order dictionary
        diag = -(-n // 64) * 64 * 3 ** dim <= val.size + val.size // 4 + 64 * 3 ** dim
        assert plans[0].m.index == (feat.IDX_DIAG if diag else feat.IDX_DICT)
        assert (plans[0].m.grid_n1, plans[0].m.grid_dim) == ((n1, dim) if diag else (0, 0))
        assert plans[1].m.index == feat.IDX_DICT and plans[1].m.grid_n1 == 0
        for filt in (None, edge, some):
            mask = None
            if filt is not None:
                idx = torch.from_numpy(np.flatnonzero(filt)).cuda()
                mask = torch.zeros((n + 31) // 32, dtype=torch.int32, device="cuda")
                feat.check(k.feat_unit_filter_mask_u64(handle.h, P(mask), n, P(idx), idx.numel()), "mask")
            out = []
            for pl in plans:
                o = [torch.full((n,), float("nan"), dtype=dt, device="cuda") for _ in range(4)]
                s = torch.zeros(2, dtype=torch.float64, device="cuda")
                if fp == "f64":
                    feat.check(k.feat_defect_f64(handle.h, pl.m, P(o[0]), P(rhs), P(x), P(mask), P(s), ws), "defect")
                    feat.check(k.feat_rj_smooth_f64(handle.h, pl.m, P(inv), P(mask), 3, 0.7, P(rhs), None, P(o[1]), P(o[2]),
                                                    P(o[3]), None, None, None, ws), "smooth")
                    feat.check(k.feat_matrix_apply_f64(handle.h, pl.m, P(o[2]), 1.5, P(x), -0.5, P(rhs)), "apply")
                else:
                    feat.check(k.feat_defect_f32(handle.h, pl.m, P(o[0]), P(rhs), P(x), P(mask), P(s), ws), "defect")
                    feat.check(k.feat_rj_smooth_f32(handle.h, pl.m, P(inv), P(mask), 3, 0.7, P(rhs), None, P(o[1]), P(o[2]),
                                                    P(o[3]), None, ws), "smooth")
                    feat.check(k.feat_apply_masked_f32(handle.h, pl.m, P(o[2]), P(x), P(mask), None, ws), "apply")
                handle.sync()
                out.append((o, float(s[0])))
            for a, b, c in zip(out[0][0], out[1][0], out[2][0]):
                assert torch.equal(a, b) and torch.equal(c, b), (fp, filt is None)
            # the norm is the same sum in another order
            assert abs(out[0][1] - out[1][1]) <= 1e-13 * out[1][1]
            assert abs(out[2][1] - out[1][1]) <= 1e-13 * out[1][1]
        for pl in plans:
            pl.close()


@pytest.mark.parametrize("dim,n1", [(2, 40), (3, 33)])
def test_odd_row_keeps_codes(feat, handle, torch_gpu, dim, n1):
    torch = torch_gpu
    k, _ = feat.libs()
    val, col, rp, _ = grid_csr(dim, n1, odd_row=True)
    n = n1 ** dim
    dev = [torch.from_numpy(a).cuda() for a in (val, col, rp)]
    plans = [feat.SellPlan(handle, *dev, n, n), feat.SellPlan(handle, *dev, n, n, diag=False)]
    assert plans[0].m.index == feat.IDX_DIAG and plans[0].m.grid_n1 == 0
    x = torch.randn(n, dtype=torch.float64, device="cuda")
    out = [torch.empty_like(x) for _ in plans]
    for pl, o in zip(plans, out):
        feat.check(k.feat_matrix_apply_f64(handle.h, pl.m, feat.ptr(o), 1.0, feat.ptr(x), 0.0, None), "apply")
    handle.sync()
    assert torch.equal(out[0], out[1])
    for pl in plans:
        pl.close()
