"""The network's gradient at sample counts around a wavefront's 16, a workgroup's 64 and the 256
workgroups of 64 samples that stride over more, against the oracle; partial buffers of the
documented size only.  Tolerances as in test_gpu_mlp.py (BF16 operands)."""
import numpy as np
import pytest

from tests.test_gpu_lafem import dev, host
from tests.test_gpu_mlp import d16, params_dev
from tests.test_mlp_oracle import NP, NPP, OW1, OB1, random_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 16384, 16385, 33000])
def test_gradient_at_edges(feat, handle, torch_gpu, oracle, n):
    print(f"mlp gradient n={n}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    p, Xb, t = random_problem(n, 40 + n)
    pd, wbf = params_dev(feat, handle, torch, p)
    Xd, td = d16(torch, Xb), dev(torch, t)
    w = min(256, -(-n // 64))
    cap = 4 * w + -(-4 * w // 32)
    part = torch.full((cap * NPP + 64,), float("nan"), dtype=torch.float32, device="cuda")
    g = torch.full((NPP,), float("nan"), dtype=torch.float32, device="cuda")
    args = (handle.h, feat.ptr(pd), feat.ptr(wbf), feat.ptr(Xd), feat.ptr(td), n, feat.ptr(part))
    assert k.feat_mlp_grad(*args, cap - 1, feat.ptr(g)) == 1   # FEAT_ERR_INVALID: buffer too small
    feat.check(k.feat_mlp_grad(*args, cap, feat.ptr(g)), "grad")
    go, gg = oracle.mlp_grad(p, Xb, t, round_bf16=True), host(g)
    assert bool(torch.isnan(part[cap * NPP:]).all())
    assert np.linalg.norm(gg[:NP] - go[:NP]) <= 1e-2 * np.linalg.norm(go[:NP])
    for a, b in ((0, 4096), (4096, 4160), (4160, 8256), (8256, 8320), (8320, 8385)):
        assert np.linalg.norm(gg[a:b] - go[a:b]) <= 3e-2 * np.linalg.norm(go[a:b]) + 1e-7, a
    assert np.isclose(gg[NPP - 1], go[NPP - 1], rtol=1e-3)
    assert not np.any(gg[OW1:OB1].reshape(64, 64)[:, 54:])
