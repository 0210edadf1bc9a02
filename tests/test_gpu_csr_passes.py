"""CSR apply against the oracle at the sizes where its passes, plain or pipelined, can go wrong:
row-blocks whose entries end on, one before and one after a pass (1024, 2048 entries), blocks
without entries between full ones, a row over many passes, one row, many row-blocks, and the mean
row lengths and numbers of row-blocks (512, 1024) on both sides of the lines between the forms."""
import numpy as np
import pytest

from oracle.pyoracle import Csr
from tests.test_gpu_lafem import dev, host, upload_csr

pytestmark = pytest.mark.gpu


def of_lengths(lens, cols, seed=3):
    rng = np.random.default_rng(seed)
    rp = np.zeros(len(lens) + 1, np.uint64)
    rp[1:] = np.cumsum(lens)
    col = rng.integers(0, cols, int(rp[-1])).astype(np.uint64)
    return Csr(len(lens), cols, rng.standard_normal(col.size), col, rp)


def blocks(totals):
    """256-row blocks with the given entry counts, one long row in each."""
    lens = []
    for i, n in enumerate(totals):
        b = np.zeros(256, np.int64)
        b[: n % 97] += 1
        b[(37 * i) % 256] += n - b.sum()
        lens += list(b)
    return lens


def mean_rows(nblocks, mean, less=0):
    """Ragged rows of nblocks blocks with exactly `mean` entries a row, `less` fewer in all."""
    lens = np.random.default_rng(7).integers(0, 2 * mean + 1, nblocks * 256)
    d = int(lens.sum()) - nblocks * 256 * mean + less
    lens[11] += max(-d, 0)
    for i in np.flatnonzero(lens > 1):
        if d <= 0:
            break
        t = min(d, int(lens[i]) - 1)
        lens[i] -= t
        d -= t
    return lens


CASES = {
    "pass_edges_piped": lambda: of_lengths(blocks([2047, 2048, 2049, 3071, 3072, 3073, 0, 4095, 4096, 4097, 1, 5119, 5120,
                                                   5121, 8191, 8193, 6144, 1025, 1023, 7167]), 900),
    "mean_10": lambda: of_lengths(mean_rows(512, 10), 4000),
    "mean_under_10": lambda: of_lengths(mean_rows(512, 10, 1), 4000),
    "mean_16_513": lambda: of_lengths(mean_rows(513, 16), 4000),
    "mean_under_16_513": lambda: of_lengths(mean_rows(513, 16, 1), 4000),
    "mean_16_1025": lambda: of_lengths(mean_rows(1025, 16), 4000),
    "mean_24_1025": lambda: of_lengths(mean_rows(1025, 24), 4000),
    "mean_32_1025": lambda: of_lengths(mean_rows(1025, 32), 4000),
    "one_row": lambda: of_lengths([1], 5),
    "no_entries": lambda: of_lengths([0] * 300, 7),
    "pass_edges": lambda: of_lengths(blocks([767, 768, 769, 1023, 1024, 1025, 2047, 2048, 2049, 0, 3071, 3072, 3073, 1, 0, 4097]), 900),
    "long_row": lambda: of_lengths([3, 50000, 0, 2] + [1] * 255, 700),
    "partial_block": lambda: of_lengths([5] * 511, 300),
    "streaming": lambda: of_lengths(np.random.default_rng(1).integers(0, 4, 6144 * 256 + 17), 1000),
    "streaming_long": lambda: of_lengths([0] * (6143 * 256) + blocks([767, 768, 769, 1536, 1537, 2304]), 500),
}


@pytest.mark.parametrize("name", list(CASES))
def test_csr_passes_bitwise(feat, handle, torch_gpu, oracle, name):
    print(f"csr passes {name}", flush=True)
    torch = torch_gpu
    k, _ = feat.libs()
    A = CASES[name]()
    if name == "pass_edges_piped":
        assert A.nnz >= 10 * A.rows
    if name.startswith("mean_"):
        mean = int("".join(c for c in name.split("_1025")[0].split("_513")[0] if c.isdigit()))
        assert A.nnz == mean * A.rows - ("under" in name)
    v, c, r = upload_csr(torch, A)
    rng = np.random.default_rng(9)
    x, y = rng.standard_normal(A.cols), rng.standard_normal(A.rows)
    xd, yd = dev(torch, x), dev(torch, y)
    rd = torch.empty_like(yd)
    P = feat.ptr
    want = oracle.csr_apply(A, x, y, 0.75, -1.25)
    for cc, rr, fn in ((c, r, k.feat_csr_apply_f64_u64), (c.int(), r.int(), k.feat_csr_apply_f64_u32)):
        rd.fill_(float("nan"))
        feat.check(fn(handle.h, P(rd), 0.75, P(xd), -1.25, P(yd), P(v), P(cc), P(rr), A.rows, A.cols, A.nnz, 0), name)
        assert np.array_equal(host(rd).view(np.uint64), want.view(np.uint64))
    x32, y32 = x.astype(np.float32), y.astype(np.float32)
    want32 = oracle.csr_apply_f32(A, x32, y32, 0.75, -1.25)
    v32, x32d, y32d = v.float(), dev(torch, x32), dev(torch, y32)
    r32 = torch.empty_like(y32d)
    for cc, rr, fn in ((c, r, k.feat_csr_apply_f32_u64), (c.int(), r.int(), k.feat_csr_apply_f32_u32)):
        r32.fill_(float("nan"))
        feat.check(fn(handle.h, P(r32), 0.75, P(x32d), -1.25, P(y32d), P(v32), P(cc), P(rr), A.rows, A.cols, A.nnz, 0), name)
        assert np.array_equal(host(r32).view(np.uint32), want32.view(np.uint32))
