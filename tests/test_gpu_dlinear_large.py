"""d-linear prolongations on both sides of the grid size from which FP64 rows load behind their
conditions (2^20 rows: 101 and 103 nodes a side in 3D), bit for bit: the weights are powers of two, so
adding the weighted neighbours one after the other in ascending order is the row's fma chain."""
import ctypes
import itertools

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n1", [(2, 1025), (3, 101), (3, 103)])
@pytest.mark.parametrize("fp", ["f64", "f32"])
def test_prolongation_rows(feat, handle, torch_gpu, dim, n1, fp):
    print(f"d-linear prolongation {dim} {n1} {fp}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    P = feat.ptr
    dt = torch.float64 if fp == "f64" else torch.float32
    nc = (n1 + 1) // 2
    g = torch.Generator(device="cuda").manual_seed(n1)
    x = torch.randn((nc,) * dim, generator=g, device="cuda", dtype=dt)
    sol = torch.randn((n1,) * dim, generator=g, device="cuda", dtype=dt)
    want = sol.clone()
    for q in itertools.product((0, 1), repeat=dim):   # parity of the fine node, slowest axis first
        s = None
        for e in itertools.product(*[(0, 1) if i else (0,) for i in q]):
            v = x[tuple(slice(e[a], nc - (q[a] - e[a])) for a in range(dim))] * 0.5 ** sum(q)
            s = v if s is None else s + v
        want[tuple(slice(i, None, 2) for i in q)] += s
    m = feat.Matrix()
    feat.check(getattr(k, "feat_matrix_dlinear_" + fp)(dim, n1, 0, ctypes.byref(m)), "dlinear")
    feat.check(getattr(k, "feat_prol_add_" + fp)(handle.h, ctypes.byref(m), P(sol), P(x), None), "prolongation")
    handle.sync()
    assert torch.equal(sol, want)
