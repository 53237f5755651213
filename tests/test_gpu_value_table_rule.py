"""Which SELL and SELD operators keep a value table: the least sizes in both
precisions and the table's limits for large operators (1024 values, or one
value per 512 rows up to 4096), the path read back in every case and products
bit for bit; infinities, NaN and signed zeros in the vector; FP32 sweeps to
the rounding of their rows."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def ragged(n, nval, most, step, seed):
    """n x n, diagonal 16 and up to `most` more entries per row at ragged columns (at most `step` apart), nval
    distinct values with the diagonal's."""
    rng = np.random.default_rng(seed)
    tab = np.unique(rng.uniform(-1.0, 1.0, 4 * nval + 16))
    rng.shuffle(tab)
    tab = tab[:nval - 1]
    rows = np.repeat(np.arange(n), rng.integers(0, most + 1, n))
    cols = rows + rng.integers(1, step, rows.size)
    rows, cols = rows[cols < n], cols[cols < n]
    key = np.unique(rows.astype(np.int64) * n + cols)
    rows, cols = key // n, key % n
    vals = tab[(np.arange(rows.size) * 7919) % tab.size]
    a = sp.csr_matrix((np.concatenate([vals, np.full(n, 16.0)]),
                       (np.concatenate([rows, np.arange(n)]), np.concatenate([cols, np.arange(n)]))), shape=(n, n))
    a.sort_indices()
    assert np.unique(a.data).size == nval
    return a


def one_level(eng, A, fmt, precision="double", sweeps=2):
    p = eng.MldPrec(device=0).init("JACOBI")
    p.set("SMOOTHER_SWEEPS", sweeps)
    p.set_format(fmt)
    return p.set_precision(precision).build(A)


@pytest.mark.parametrize("n,nval,fmt,precision,taken", [
    (32767, 7, "sell", "double", False), (32768, 7, "sell", "double", True), (98303, 7, "sell", "mixed", False),
    (98304, 7, "sell", "mixed", True), (98303, 7, "seld", "mixed", False), (98305, 7, "seld", "mixed", True)])
def test_least_rows(eng, n, nval, fmt, precision, taken):
    p = one_level(eng, ragged(n, nval, 9, 900, n), fmt, precision)
    assert p.op_bytes_form(0, "A") == fmt.upper() + ("+values" if taken else "")


# values with the padding's zero: 1024; 1050624 / 512 = 2052; 4096.  A word's bits: SELL's columns leave 11 of them
# from 1048577 columns on and 10 from 2097153 on, SELD's steps 16.
@pytest.mark.parametrize("fmt", ["sell", "seld128"])
@pytest.mark.parametrize("n,most,nval,fits", [
    (65000, 9, 1023, True), (65000, 9, 1024, False), (1048576, 3, 2047, True), (1048576, 3, 2048, False),
    (1050624, 3, 2051, True), (1050624, 3, 2052, False), (2097152, 2, 4095, True), (2100000, 2, 4096, False)])
def test_limits(eng, orc, fmt, n, most, nval, fits):
    print(f"[value table rule] {fmt} n {n} values {nval}", flush=True)
    A = ragged(n, nval, most, 5000, n + nval)
    p = one_level(eng, A, fmt)
    taken = fits and (fmt != "sell" or nval + 1 <= 1 << (32 - (n - 1).bit_length()))
    assert p.op_bytes_form(0, "A") == fmt[:4].upper() + ("+values" if taken else "")
    x = np.random.default_rng(n).standard_normal(n)
    y = torch.zeros(n, dtype=torch.float64, device="cuda:0")
    p.level_spmv(0, "A", dev(x), y)
    assert (y.cpu().numpy() == orc.Csr.from_scipy(A).spmv(x)).all()


@pytest.mark.parametrize("fmt", ["sell", "seld"])
@pytest.mark.parametrize("n,nval", [(40003, 50), (98304, 1000)])
def test_special_values(eng, orc, fmt, n, nval):
    """Padding multiplies a zero with the row's own column (SELL) or those behind its last one (SELD), as in the
    products without a table: rows that see a special value only there are left out."""
    A = ragged(n, nval, 9, 300, n + nval)
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n)
    at = np.unique(rng.integers(0, n, 60))
    x[at] = np.array([np.inf, -np.inf, np.nan, -0.0, 0.0])[np.arange(at.size) % 5]
    p = one_level(eng, A, fmt)
    assert p.op_bytes_form(0, "A") == fmt.upper() + "+values"
    y = torch.zeros(n, dtype=torch.float64, device="cuda:0")
    p.level_spmv(0, "A", dev(x), y)
    y = y.cpu().numpy()
    with np.errstate(all="ignore"):
        ref = orc.Csr.from_scipy(A).spmv(x)
    bad = ~np.isfinite(x)
    last = A.indices[A.indptr[1:] - 1]
    behind = np.zeros(n, bool)
    for k in range(1, 11):
        behind |= bad[np.minimum(last + k, n - 1)]
    keep = ~(bad | behind)
    assert keep.sum() > 0.9 * n and not np.isfinite(ref[keep]).all()
    assert (np.isnan(y) == np.isnan(ref))[keep].all()
    ok = keep & ~np.isnan(ref)
    assert (y[ok].view(np.int64) == ref[ok].view(np.int64)).all()


@pytest.mark.parametrize("fmt", ["sell", "seld"])
@pytest.mark.parametrize("n,nval", [(98304, 3), (120001, 900)])
def test_fp32_sweeps(eng, fmt, n, nval):
    """Three sweeps: the products with ND D and with ND, both with tables."""
    A = ragged(n, nval, 9, 900, n + nval)
    x = np.random.default_rng(n).standard_normal(n)
    nd = (A - sp.diags(A.diagonal())).tocsr()
    w = int(np.diff(nd.indptr).max())
    for precision, ulp in (("double", 2.0 ** -53), ("mixed", 2.0 ** -24)):
        p = one_level(eng, A, fmt, precision, sweeps=3)
        assert p.op_bytes_form(0, "ND") == fmt.upper() + "+values"
        y = p.apply(dev(x)).cpu().numpy()
        t, bound = x / 16.0, 0.0
        for _ in range(2):
            # every input and operation rounded once: values, d and ND D (3), x (1), w products and sums, the
            # subtraction and the last product (2); and what the sweep before was off
            bound = (abs(nd) @ (bound * np.ones(n)) + (w + 8) * ulp * (np.abs(x) + abs(nd) @ np.abs(t))) / 16.0
            t = (x - nd @ t) / 16.0
        assert (np.abs(y - t) <= bound).all(), precision
