"""Banded plans with symmetric values read half of them from the neighbours' rows: bit-identical
to the plain plan, on symmetric matrices and on matrices with one entry off by one bit (which
keep reading every slot), at grid sizes around the 256-row chunks."""
import numpy as np
import pytest

from tests.test_gpu_stencil_march import grid_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("symmetric", [True, False])
@pytest.mark.parametrize("dim,n1", [(2, 6), (2, 16), (2, 17), (2, 100), (3, 3), (3, 5), (3, 7), (3, 20)])
def test_symmetric_banded_bitwise(feat, handle, torch_gpu, dim, n1, symmetric):
    print(f"banded dim={dim} n1={n1} symmetric={symmetric}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    P = feat.ptr
    _, col, rp, _ = grid_csr(dim, n1)
    n = n1 ** dim
    row = np.repeat(np.arange(n), np.diff(rp))
    # one value per unordered pair: (i, j) and (j, i) get the same
    lo, hi = np.minimum(row, col), np.maximum(row, col)
    _, pair = np.unique(lo * n + hi, return_inverse=True)
    val = np.random.default_rng(n1).uniform(-1, 1, pair.max() + 1)[pair]
    if not symmetric:
        e = int(rp[n // 2])
        val[e] = np.float64(np.float16(val[e])) + 0.25   # differs in every precision
    dev = [torch.from_numpy(a).cuda() for a in (val, col, rp)]
    x64, rhs64 = (torch.from_numpy(v).cuda() for v in np.random.default_rng(1).standard_normal((2, n)))
    keep, ws = feat.reduce_ws(torch, "cuda")
    for fp in ("f64", "f32", "f16"):
        band = feat.SellPlan(handle, *dev, n, n, fp=fp)
        plain = feat.SellPlan(handle, *dev, n, n, fp=fp, banded=False)
        if band.m.format != feat.FMT_BANDED:   # few enough values for a dictionary
            assert n < 60
            continue
        assert band.m.grid_n1 == (n1 if symmetric else 0)
        dt = torch.float64 if fp == "f64" else torch.float32
        x, rhs = x64.to(dt), rhs64.to(dt)
        out = []
        for pl in (band, plain):
            d, r = torch.empty_like(x), torch.empty_like(x)
            s = torch.zeros(2, dtype=torch.float64, device="cuda")
            if fp == "f64":
                feat.check(k.feat_defect_f64(handle.h, pl.m, P(d), P(rhs), P(x), None, P(s), ws), "defect")
                feat.check(k.feat_matrix_apply_f64(handle.h, pl.m, P(r), -0.5, P(x), 2.0, P(rhs)), "apply")
            else:
                feat.check(k.feat_defect_f32(handle.h, pl.m, P(d), P(rhs), P(x), None, P(s), ws), "defect")
                feat.check(k.feat_apply_masked_f32(handle.h, pl.m, P(r), P(x), None, None, ws), "apply")
            handle.sync()
            out.append((d, r, s))
        for a, b in zip(*out):
            assert torch.equal(a, b), fp
        band.close()
        plain.close()
