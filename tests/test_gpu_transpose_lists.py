"""The transposed CSR apply's column lists against the oracle, bit for bit, at the sizes where they
can go wrong: list lengths around 64, what shares a workgroup (192) and what one holds (1024),
many long columns, lists whose parts by entry number do not fit (clustered entries), dense columns, columns without entries, repeated columns in a row, unsorted rows, rows
without entries, tiles of entries that start and end inside a row."""
import numpy as np
import pytest

from oracle.pyoracle import Csr
from tests.helpers import random_csr
from tests.test_gpu_lafem import dev, host, upload_csr

pytestmark = pytest.mark.gpu


def by_columns(rng, rows, lens):
    """Entries so that column c holds lens[c], in random rows (repeats allowed), unsorted."""
    col = np.repeat(np.arange(len(lens)), lens)
    row = rng.integers(0, rows, col.size)
    order = np.lexsort((rng.random(col.size), row))
    rp = np.zeros(rows + 1, np.uint64)
    rp[1:] = np.cumsum(np.bincount(row, minlength=rows))
    return Csr(rows, len(lens), rng.standard_normal(col.size), col[order].astype(np.uint64), rp)


def clustered(rng):
    """Column 0: 3000 entries in a row, and one far behind them; column 1: 5000 spread evenly."""
    mid = np.concatenate([rng.integers(2, 300, 60000), np.full(5000, 1)])
    rng.shuffle(mid)
    col = np.concatenate([np.zeros(3000, np.int64), mid, [0]])
    rp = np.concatenate([[0], np.sort(rng.integers(0, col.size, 199)), [col.size]]).astype(np.uint64)
    return Csr(200, 300, rng.standard_normal(col.size), col.astype(np.uint64), rp)


CASES = {
    "clustered": clustered,
    "around_192": lambda g: by_columns(g, 700, [191, 192, 193, 194, 0, 190] * 9),
    "few_columns": lambda g: by_columns(g, 700, [192, 193, 1, 100, 64]),
    "many_long": lambda g: by_columns(g, 3000, [2900] * 70),
    "many_medium": lambda g: by_columns(g, 3000, [65, 70, 200] * 500),
    "long_steps": lambda g: by_columns(g, 9000, [1025, 2047, 3, 4097, 0, 8193, 1026] * 3),
    "one": lambda g: by_columns(g, 1, [1]),
    "short": lambda g: by_columns(g, 500, [0, 1, 2, 63, 64] * 40),
    "around_64": lambda g: by_columns(g, 300, [63, 64, 65, 66, 127, 128, 129] * 19),
    "around_cap": lambda g: by_columns(g, 5000, [1023, 5, 1024, 0, 1025, 64, 2048, 2049, 1]),
    "dense": lambda g: by_columns(g, 40000, [30000] + [3] * 200),
    "cap_filled": lambda g: by_columns(g, 900, [32] * 64 + [33] * 64 + [31, 64] * 32),
    "empty_rows": lambda g: by_columns(g, 30000, [7] * 900),
    "one_long_row": lambda g: random_csr(g, 40, 20000, 0, 5, [(7, 15000)]),
    "random": lambda g: random_csr(g, 3000, 1700, 0, 30, [(5, 1600)]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_transposed_lists_bitwise(feat, handle, torch_gpu, oracle, name):
    print(f"transposed lists {name}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    rng = np.random.default_rng(12)
    A = CASES[name](rng)
    v, c, r = upload_csr(torch, A)
    x, y = rng.standard_normal(A.rows), rng.standard_normal(A.cols)
    xd, yd = dev(torch, x), dev(torch, y)
    for a, b in [(1.0, 0.0), (-0.7, 1.0)]:
        want = oracle.csr_apply(A, x, y, a, b, transposed=True)
        rd = torch.full((A.cols,), 7.0, dtype=torch.float64, device="cuda")
        args = (handle.h, feat.ptr(rd), a, feat.ptr(xd), b, feat.ptr(yd), feat.ptr(v), feat.ptr(c), feat.ptr(r), A.rows,
                A.cols, A.nnz)
        for again in range(2):
            feat.check(k.feat_csr_apply_f64_u64(*args, 1), "transposed")
            assert np.array_equal(host(rd).view(np.uint64), want.view(np.uint64)), (a, b, again)
        rd.fill_(7.0)
        feat.check(k.feat_csr_apply_transposed_noalloc_f64_u64(*args), "noalloc")
        assert np.array_equal(host(rd).view(np.uint64), want.view(np.uint64)), (a, b)
    yd.copy_(dev(torch, y))   # r == y
    feat.check(k.feat_csr_apply_f64_u64(handle.h, feat.ptr(yd), 0.5, feat.ptr(xd), 2.0, feat.ptr(yd), feat.ptr(v),
                                        feat.ptr(c), feat.ptr(r), A.rows, A.cols, A.nnz, 1), "transposed in place")
    want = oracle.csr_apply(A, x, y, 0.5, 2.0, transposed=True)
    assert np.array_equal(host(yd).view(np.uint64), want.view(np.uint64))
