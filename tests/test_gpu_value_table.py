"""SELL and SELD operators of few distinct values (one 32-bit word per entry,
values looked up in a table): products bit for bit against the oracle's
sequential ones, at 1 to 1024 distinct values (and 1025, which keep the
arrays), around the least size and whole workgroups; FP32 products to the
rounding of their rows; hierarchies and their solves."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def tables(capfd):
    return [q for q in capfd.readouterr().err.splitlines() if "distinct values" in q]


def ragged(n, nval, step, seed):
    """n x n, diagonal and up to 11 more entries per row at ragged columns (at
    most `step` apart), nval distinct values with those of the diagonal (and
    the padding's zero)."""
    rng = np.random.default_rng(seed)
    tab = np.unique(rng.uniform(-1.0, 1.0, 8 * nval + 16))[: max(nval - 1, 0)]
    rng.shuffle(tab)
    tab = np.concatenate([[16.0], tab])[:nval]
    cnt = rng.integers(0, 12, n)
    rows = np.repeat(np.arange(n), cnt)
    cols = rows + rng.integers(1, step, rows.size)
    keep = cols < n
    rows, cols = rows[keep], cols[keep]
    key = np.unique(rows.astype(np.int64) * n + cols)
    rows, cols = key // n, key % n
    vals = tab[(np.arange(rows.size) * 7919) % nval]
    a = sp.csr_matrix((np.concatenate([vals, np.full(n, 16.0)]),
                       (np.concatenate([rows, np.arange(n)]), np.concatenate([cols, np.arange(n)]))), shape=(n, n))
    a.sort_indices()
    return a


@pytest.mark.parametrize("fmt", ["sell", "seld128"])
@pytest.mark.parametrize("n,nval,step,packed", [
    (32768, 1, 40, True), (32769, 2, 3000, True), (33000, 255, 5000, True), (40001, 1023, 700, True),
    (32767, 3, 40, False), (50000, 1025, 900, False), (1048577, 5, 60000, True)])
def test_products(eng, orc, monkeypatch, capfd, fmt, n, nval, step, packed):
    """1023 values and the padding's zero fill the table."""
    monkeypatch.setenv("MLD_VERBOSE", "1")
    print(f"[value table] {fmt} n {n} values {nval} step {step}", flush=True)
    A = ragged(n, nval, step, n + nval)
    tables(capfd)
    p = eng.MldPrec(device=0).init("JACOBI")
    p.set_format(fmt)
    p.build(A)
    assert p.op_format(0, "A")["fmt"] == fmt[:4].upper()
    assert any(f"{n} x {n} operator" in q for q in tables(capfd)) == packed
    x = np.random.default_rng(n).standard_normal(n)
    y = torch.zeros(n, dtype=torch.float64, device="cuda:0")
    p.level_spmv(0, "A", dev(x), y)
    assert (y.cpu().numpy() == orc.Csr.from_scipy(A).spmv(x)).all()


@pytest.mark.parametrize("idim", [64, 97, 101])
def test_hierarchy(eng, orc, monkeypatch, capfd, idim):
    """Level 1 of Poisson: transfers and operators take the table where their
    layout is SELL or SELD; every product as the sequential one, and solves in
    both precisions reach the residual that they report."""
    monkeypatch.setenv("MLD_VERBOSE", "1")
    print(f"[value table hierarchy] {idim}", flush=True)
    A = orc.gen_pde3d(idim).to_scipy()
    b = np.random.default_rng(idim).standard_normal(A.shape[0])
    for precision in ("double", "mixed"):
        p = eng.MldPrec(device=0).init("ML")
        for k, v in (("SMOOTHER_TYPE", "L1-JACOBI"), ("SMOOTHER_SWEEPS", 2), ("AGGR_THRESH", 0.0),
                     ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 200), ("COARSE_SOLVE", "BJAC"),
                     ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
            p.set(k, v)
        tables(capfd)
        p.set_precision(precision).build(A)
        assert len(tables(capfd)) >= 1
        if precision == "double":
            for what in ("A", "P", "R", "ND"):
                m = p.level_csr(1, what)
                f = p.op_format(1, what)
                x = np.random.default_rng(7).standard_normal(m.shape[1])
                y = torch.zeros(m.shape[0], dtype=torch.float64, device="cuda:0")
                p.level_spmv(1, what, dev(x), y)
                ref = orc.Csr.from_scipy(m).spmv(x)
                if f["fmt"] in ("SELL", "SELD"):
                    assert (y.cpu().numpy() == ref).all(), what
                else:
                    assert np.abs(y.cpu().numpy() - ref).max() <= 1e-13 * np.abs(ref).max(), what
        x, it, err = eng.psb_krylov("CG", A, p, dev(b), eps=1e-9)
        assert err <= 1e-9
        assert np.linalg.norm(b - A @ x.cpu().numpy()) <= 1.01e-9 * np.linalg.norm(b)
