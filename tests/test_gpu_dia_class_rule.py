"""Which banded operators keep a class byte per row: those of at most 256
distinct rows whose stored values take at least 7 MB.  The path is read back
in every case; products bit for bit as the stored diagonals give them (numpy,
one diagonal after the other), with infinities, NaN and signed zeros in the
vector too, and FP32 sweeps to the rounding of their rows."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def diagonals(a):
    """(offsets, values by diagonal, 0 where a row has no such entry) of a CSR matrix."""
    c = a.tocoo()
    offs = np.unique(c.col - c.row)
    v = np.zeros((offs.size, a.shape[0]))
    v[np.searchsorted(offs, c.col - c.row), c.row] = c.data
    return offs, v


def product(offs, v, x):
    """The stored form's arithmetic: every diagonal in turn, outside columns at the ends of x."""
    n = v.shape[1]
    i, acc = np.arange(n), np.zeros(n, v.dtype)
    with np.errstate(all="ignore"):
        for k, o in enumerate(offs):
            acc = acc + v[k] * x[np.clip(i + o, 0, n - 1)]
    return acc


def classes(offs, v):
    return np.unique(v.T, axis=0).shape[0]


def banded(n, offs, ncls, seed):
    """n x n, constant diagonal (unless it is the only one), exactly ncls distinct rows (the rows at the two ends,
    which lack diagonals, are some of them)."""
    rng = np.random.default_rng(seed)
    ends = sum(len({min(max(abs(o), 0), n) for o in offs if o * s > 0}) for s in (-1, 1))
    edge = np.unique([abs(o) for o in offs if o < 0])[::-1]
    inner = ncls - ends
    assert inner >= 1
    tab = rng.uniform(-1.0, 1.0, (inner, len(offs)))
    if len(offs) > 1:
        tab[:, list(offs).index(0)] = 9.0
    lo = int(edge[0]) if edge.size else 0
    hi = n - max(max(offs), 0)
    c = (np.arange(n, dtype=np.int64) * 7919 // 3) % inner
    c[n // 3: 2 * n // 3] = 0
    c[:lo] = 0
    c[hi:] = 0
    data, i = [], np.arange(n)
    for k, o in enumerate(offs):
        q = i[max(0, -o): min(n, n - o)]
        data.append((q, q + o, tab[c[q], k]))
    r, col, v = (np.concatenate(t) for t in zip(*data))
    a = sp.csr_matrix((v, (r, col)), shape=(n, n))
    a.sort_indices()
    return a


# n x offsets x distinct rows x takes the form (7 MB: 291667 rows of 3, 875000 of 1, 125000 of 7)
CASES = [
    (300001, (-1, 0, 1), 255, True), (300000, (-1, 0, 1), 256, True), (300001, (-1, 0, 1), 257, False),
    (875001, (0,), 256, True), (875001, (0,), 257, False), (874999, (0,), 3, False),
    (125003, (-311, -17, -1, 0, 1, 17, 311), 256, True), (125003, (-311, -17, -1, 0, 1, 17, 311), 257, False),
    (124999, (-311, -17, -1, 0, 1, 17, 311), 40, False), (131072, (-500, -9, -3, 0, 1, 2, 11, 40), 200, True)]


@pytest.mark.parametrize("n,offs,ncls,taken", CASES)
def test_limits(eng, n, offs, ncls, taken):
    print(f"[class rule] n {n} offsets {offs} rows {ncls}", flush=True)
    A = banded(n, offs, ncls, n + ncls)
    o, v = diagonals(A)
    assert tuple(o) == offs and classes(o, v) == ncls
    p = eng.MldPrec(device=0).init("JACOBI")
    p.set("SMOOTHER_SWEEPS", 2)
    p.build(A)
    assert p.op_bytes_form(0, "A") == ("DIA+rows" if taken else "DIA")
    rng = np.random.default_rng(n)
    for special in (False, True):
        x = rng.standard_normal(n)
        if special:
            at = rng.integers(0, n, 40)
            x[at] = np.array([np.inf, -np.inf, np.nan, -0.0, 0.0])[np.arange(40) % 5]
            x[[0, n - 1]] = -0.0, np.inf
        y = torch.zeros(n, dtype=torch.float64, device="cuda:0")
        p.level_spmv(0, "A", dev(x), y)
        ref, y = product(o, v, x), y.cpu().numpy()
        assert (np.isnan(ref) == np.isnan(y)).all()
        ok = ~np.isnan(ref)
        assert (ref[ok].view(np.int64) == y[ok].view(np.int64)).all()  # signs of zeros too


@pytest.mark.parametrize("n,offs,ncls", [
    (350001, (-1, 0, 1), 9), (875001, (-1, 0, 1), 256), (437500, (-2, -1, 0, 1, 2), 257),
    (300001, (-311, -17, -1, 0, 1, 17, 311), 256)])
def test_sweeps(eng, n, offs, ncls):
    """Two sweeps in FP64 and FP32: d (x - ND D x), the diagonal from the class."""
    A = banded(n, offs, ncls, n + ncls)
    x = np.random.default_rng(n).standard_normal(n)
    d = 1.0 / A.diagonal()
    nd = (A - sp.diags(A.diagonal())).tocsr()
    w = len(offs) - 1
    for precision, size, ulp in (("double", 8, 2.0 ** -53), ("mixed", 4, 2.0 ** -24)):
        p = eng.MldPrec(device=0).init("JACOBI")
        p.set("SMOOTHER_SWEEPS", 2)
        p.set_precision(precision).build(A)
        taken = w * n * size >= 7e6 and ncls <= 256
        assert p.op_bytes_form(0, "ND") == ("DIA+rows" if taken else "DIA"), precision
        y = p.apply(dev(x)).cpu().numpy()
        ref = d * (x - nd @ (d * x))
        # every input and operation rounded once: values, d and ND D of d (3), x (1), w products and sums, the
        # subtraction and the last product (2)
        bound = (w + 8) * ulp * np.abs(d) * (np.abs(x) + abs(nd) @ np.abs(d * x))
        assert (np.abs(y - ref) <= bound).all(), precision


@pytest.mark.parametrize("idim,precision,taken", [
    (33, "double", False), (48, "double", False), (56, "double", True), (33, "mixed", False), (56, "mixed", False),
    (72, "mixed", True)])
def test_small_levels_keep_their_values(eng, orc, idim, precision, taken):
    A = orc.gen_pde3d(idim).to_scipy()
    p = eng.MldPrec(device=0).init("JACOBI")
    p.set("SMOOTHER_SWEEPS", 2)
    p.set_precision(precision).build(A)
    assert p.op_bytes_form(0, "A") == ("DIA+rows" if taken else "DIA")
