"""The first iterate of an FP32 smoother formed by the kernel that produces its right-hand side
(defect, masked apply, conversion from FP64): the smoother then gives the bits of the one that
forms the iterate itself, with random, zero (skip rule) and NaN right-hand sides, for even and odd
step counts (either ping-pong buffer), on grid and general plans."""
import numpy as np
import pytest

from tests.test_gpu_lafem import dev, host, upload_csr
from tests.test_gpu_solver import mask_of, q1_level

pytestmark = pytest.mark.gpu


def same(a, b):
    assert np.array_equal(np.isnan(a), np.isnan(b))
    ok = ~np.isnan(a)
    assert np.array_equal(a[ok].view(np.uint32), b[ok].view(np.uint32))


@pytest.mark.parametrize("steps", [2, 3])
@pytest.mark.parametrize("rhs_kind", ["random", "zero", "nan"])
@pytest.mark.parametrize("plain", [False, True])
def test_first_iterate_f32_bitwise(feat, handle, torch_gpu, steps, rhs_kind, plain):
    print(f"FP32 first iterate steps={steps} {rhs_kind} plain={plain}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    P = feat.ptr
    keep, ws = feat.reduce_ws(torch, "cuda")
    q, A = q1_level(feat, 3, 3)
    n = q["n"]
    v, c, r = upload_csr(torch, A)
    plan = feat.SellPlan(handle, v, c, r, n, n, fp="f32", dict=not plain, banded=not plain)
    m = mask_of(torch, feat, handle, n, q["filt"])
    rng = np.random.default_rng(50 + steps)
    inv = dev(torch, (0.3 + rng.random(n)).astype(np.float32))
    b64 = rng.standard_normal(n)
    x0 = rng.standard_normal(n).astype(np.float32)
    if rhs_kind == "zero":
        b64[:] = 0.0
        x0[:] = 0.0
    elif rhs_kind == "nan":
        b64[n // 2] = np.nan
    bd, xd = dev(torch, b64), dev(torch, x0)
    sol0 = rng.standard_normal(n).astype(np.float32)

    def vec():
        return torch.zeros(n, dtype=torch.float32, device="cuda")

    try:
        outs = []
        for first in (False, True):
            fn = k.feat_rj_smooth_from1_f32 if first else k.feat_rj_smooth_f32
            got = []
            # conversion, then pre-smoothing with its final defect
            nrm = torch.zeros(1, dtype=torch.float64, device="cuda")
            feat.check(k.feat_dot_f64(handle.h, P(nrm), P(bd), P(bd), n), "norm")
            rhs, x, tmp, d = vec(), vec(), vec(), vec()
            x1 = x if steps & 1 else tmp
            if first:
                feat.check(k.feat_convert_first_f64_f32(handle.h, P(rhs), P(bd), n, P(inv), P(m), 0.8, P(x1)), "convert")
            else:
                feat.check(k.feat_convert_f64_f32(handle.h, P(rhs), P(bd), n), "convert")
            feat.check(fn(handle.h, plan.m, P(inv), P(m), steps, 0.8, P(rhs), P(nrm), P(x), P(tmp), P(d), None, ws), "pre")
            handle.sync()
            got += [host(x), host(d)]
            # masked apply, then pre-smoothing
            rr, x2, tmp2, d2 = vec(), vec(), vec(), vec()
            src = rhs if rhs_kind == "nan" else xd
            x1 = x2 if steps & 1 else tmp2
            if first:
                feat.check(k.feat_apply_masked_first_f32(handle.h, plan.m, P(rr), P(src), P(m), P(nrm), P(inv), 0.8, P(x1),
                                                         ws), "masked")
            else:
                feat.check(k.feat_apply_masked_f32(handle.h, plan.m, P(rr), P(src), P(m), P(nrm), ws), "masked")
            feat.check(fn(handle.h, plan.m, P(inv), P(m), steps, 0.8, P(rr), P(nrm), P(x2), P(tmp2), P(d2), None, ws), "pre")
            handle.sync()
            got += [host(x2), host(d2)]
            # defect, then post-smoothing accumulated into sol
            d3, cor, tmp3, sol = vec(), vec(), vec(), dev(torch, sol0)
            x1 = cor if steps & 1 else tmp3
            if first:
                feat.check(k.feat_defect_first_f32(handle.h, plan.m, P(d3), P(rhs), P(xd), P(m), P(nrm), P(inv), 0.8, P(x1),
                                                   ws), "defect")
            else:
                feat.check(k.feat_defect_f32(handle.h, plan.m, P(d3), P(rhs), P(xd), P(m), P(nrm), ws), "defect")
            feat.check(fn(handle.h, plan.m, P(inv), P(m), steps, 0.8, P(d3), P(nrm), P(cor), P(tmp3), None, P(sol), ws),
                       "post")
            handle.sync()
            got += [host(d3), host(sol)]
            outs.append(got)
        for a, b in zip(*outs):
            same(a, b)
    finally:
        plan.close()
