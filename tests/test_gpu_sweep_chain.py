"""Triangular sweeps run as one launch (chained level sets): SOR / SSOR / ILU(0) against the
oracle's sequential sweeps, bit for bit, at the sizes where the chain can go wrong: one row,
slices of 63 / 64 / 65 rows, one level, levels of one row, rows longer than the entries held
in registers, levels of more slices than waves, dependencies farther apart than the LDS ring
holds (per-level launches), and positions that wrap around the ring.  Where the chain's padding
or its widest levels would cost more than it gains the sweeps keep their launches."""
import numpy as np
import pytest

from oracle.pyoracle import Csr
from tests.test_gpu_smoothers import upload
from tests.test_smoothers_oracle import dominant, q1_csr

pytestmark = pytest.mark.gpu


def from_rows(rows):
    """CSR of {column: value} rows with their diagonals."""
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.uint64)
    col = np.concatenate([sorted(r) for r in rows]).astype(np.uint64)
    val = np.concatenate([[r[c] for c in sorted(r)] for r in rows])
    return Csr(len(rows), len(rows), val, col, rp)


def banded(n, offsets, seed=1):
    """Symmetric pattern with entries at the given offsets, diagonally dominant."""
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(n):
        r = {i + s * o: rng.uniform(-1, 1) for o in offsets for s in (-1, 1) if 0 <= i + s * o < n}
        r[i] = 2.0 * len(offsets) + 1.0
        rows.append(r)
    return from_rows(rows)


def matrices(feat):
    rng = np.random.default_rng(5)
    return {
        "one_row": lambda: banded(1, []),
        "diagonal_65": lambda: banded(65, []),
        "chain_200": lambda: banded(200, [1]),
        "slices_63": lambda: banded(63 * 4, [63]),
        "slices_64": lambda: banded(64 * 4, [64]),
        "slices_65": lambda: banded(65 * 4, [65]),
        "long_rows": lambda: banded(600, list(range(1, 40, 2)) + [97]),
        "wide_levels": lambda: banded(6000, [1500, 2999]),
        "random": lambda: dominant(rng, 2000, max_len=15),
        "far": lambda: banded(40000, [17000]),
        "q1_2d_l6": lambda: q1_csr(feat, 2, 6),
        "q1_3d_l5": lambda: q1_csr(feat, 3, 5),
    }


@pytest.mark.parametrize("name", ["one_row", "diagonal_65", "chain_200", "slices_63", "slices_64", "slices_65", "long_rows",
                                  "wide_levels", "random", "far", "q1_2d_l6", "q1_3d_l5"])
def test_chained_sweeps_equal_sequential(feat, oracle, handle, torch_gpu, name):
    print(f"chained sweeps {name}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    A = matrices(feat)[name]()
    keep, desc = upload(feat, torch, A)
    x = np.random.default_rng(8).standard_normal(A.rows)
    xd = torch.from_numpy(x).cuda()
    y = torch.full_like(xd, float("nan"))
    plan = feat.SorPlan(handle, desc)
    chain = name != "far"
    assert plan.chained()[0] == plan.chained(True)[0] == chain
    for omega in (1.0, 1.3):
        plan.sor(y, xd, omega)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), oracle.sor_generic_apply(A, omega, x))
        y.fill_(float("nan"))
        plan.ssor(y, xd, omega)
        feat.check(k.feat_scale_f64(handle.h, feat.ptr(y), feat.ptr(y), omega * (2.0 - omega), A.rows), "scale")
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), oracle.sor_generic_apply(A, omega, x, ssor=True))
    plan.close()
    ilu = feat.IluPlan(handle, desc)
    assert ilu.chained()[0] == ilu.chained(True)[0] == chain
    f = oracle.ilu0_factor(A)
    want = oracle.ilu0_apply(A, f, x)
    ilu.apply(y, xd)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), want)
    ilu.apply(xd, xd)
    torch.cuda.synchronize()
    assert np.array_equal(xd.cpu().numpy(), want)
    ilu.close()


def leveled(nlevels, width, k, first=0, wide_row=0, seed=3):
    """Levels of `width` rows, each row with k entries in the two levels before it, after `first`
    rows of their own in the first level; one row of `wide_row` entries in the middle."""
    n = first + nlevels * width
    rng = np.random.default_rng(seed)
    rows = []
    for i in range(n):
        r = {i - o: rng.uniform(-1, 1) for o in range(width, width + k) if i - o >= first}
        if wide_row and i == n // 2:
            r.update({i - o: rng.uniform(-1, 1) for o in range(width, width + wide_row)})
        rows.append(r)
    for i in range(n):
        for j in [c for c in rows[i] if c < i]:
            rows[j][i] = rng.uniform(-1, 1)
    for i, r in enumerate(rows):
        r[i] = len(r) + 1.0
    return from_rows(rows)


# matrix, whether the sweeps are chained, most device bytes a row of the chain of one direction
BOUNDS = {
    "levels_of_one_row": (lambda: leveled(4000, 1, 1), True, 6100),
    "too_many_of_one_row": (lambda: leveled(30000, 1, 1), False, 0),
    "one_wide_row": (lambda: leveled(3000, 1, 1, wide_row=20), True, 6400),
    "levels_of_1500": (lambda: leveled(20, 1500, 3), True, 110),
    "levels_of_4000": (lambda: leveled(6, 4000, 3), False, 0),
    "levels_of_1500_long_rows": (lambda: leveled(12, 1500, 20), False, 0),
    "wide_first_level": (lambda: leveled(40, 64, 3, first=100000), False, 0),
    "first_level_among_many": (lambda: leveled(400, 64, 3, first=20000), True, 110),
}


@pytest.mark.parametrize("name", list(BOUNDS))
def test_chain_bounds(feat, oracle, handle, torch_gpu, name):
    print(f"chain bounds {name}", flush=True)
    torch = torch_gpu
    make, chain, per_row = BOUNDS[name]
    A = make()
    keep, desc = upload(feat, torch, A)
    x = np.random.default_rng(8).standard_normal(A.rows)
    xd = torch.from_numpy(x).cuda()
    y = torch.full_like(xd, float("nan"))
    plan, ilu = feat.SorPlan(handle, desc), feat.IluPlan(handle, desc)
    for p in (plan, ilu):
        for backward in (False, True):
            on, size = p.chained(backward)
            assert on == chain and size <= per_row * A.rows, (on, size / A.rows)
    plan.sor(y, xd, 1.2)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), oracle.sor_generic_apply(A, 1.2, x))
    ilu.apply(y, xd)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy(), oracle.ilu0_apply(A, oracle.ilu0_factor(A), x))
    plan.close()
    ilu.close()
