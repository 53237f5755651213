"""Banded operators with few distinct rows (one byte per row names its class):
products bit for bit against the oracle's sequential ones, at odd and even
sizes around the least size that takes this form and around whole workgroups,
with 1 to 256 classes (and 257 and 300, which keep the stored diagonals), 1 to
8 diagonals; Jacobi sweeps (the diagonal taken from the class) to 1e-13."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def banded(n, offs, ncls, seed):
    """n x n, diagonals offs, row i's values those of class (7919 i / 3) mod
    ncls, but of class 0 in the middle third."""
    rng = np.random.default_rng(seed)
    tab = rng.uniform(-1.0, 1.0, (ncls, len(offs)))
    tab[:, list(offs).index(0)] = 4.0 + rng.uniform(0.0, 1.0, ncls)
    c = (np.arange(n, dtype=np.int64) * 7919 // 3) % ncls
    c[n // 3: 2 * n // 3] = 0  # a long stretch of one class
    data = []
    for k, o in enumerate(offs):
        v = np.zeros(n)
        i = np.arange(max(0, -o), min(n, n - o))
        v[i + o] = tab[c[i], k]
        data.append(v)
    a = sp.dia_matrix((np.array(data), offs), shape=(n, n)).tocsr()
    a.sort_indices()
    return a


@pytest.mark.parametrize("n,offs,ncls", [
    (32768, (-1, 0, 1), 1), (32769, (-1, 0, 1), 3), (33793, (-190, -1, 0, 1, 190), 7),
    (40001, (-1000, -31, -1, 0, 1, 31, 1000), 256), (40000, (-1000, -31, -1, 0, 1, 31, 1000), 255),
    (40003, (-1000, -31, -1, 0, 1, 31, 1000), 257), (34816, (0,), 40), (36864, (-5, 0), 2),
    (37889, (-9, -3, -2, 0, 1, 2, 11, 500), 100), (40000, (-2, 0, 3), 300), (32767, (-1, 0, 1), 3)])
def test_dia_classes(eng, orc, n, offs, ncls):
    print(f"[dia classes] n {n} offsets {offs} classes {ncls}", flush=True)
    A = banded(n, offs, ncls, n + ncls)
    p = eng.MldPrec(device=0).init("JACOBI")
    p.set("SMOOTHER_SWEEPS", 2)
    p.build(A)
    assert p.op_format(0, "A")["fmt"] == "DIA"
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n)
    for what in ("A", "ND"):
        m = p.level_csr(0, what)
        if m.nnz == 0:
            continue
        y = torch.zeros(n, dtype=torch.float64, device="cuda:0")
        p.level_spmv(0, what, dev(x), y)
        assert (y.cpu().numpy() == orc.Csr.from_scipy(m).spmv(x)).all(), what
    nd, d = p.level_csr(0, "ND"), p.dv(0)
    for sweeps, beta in ((2, 0), (2, 1), (3, 0), (4, 1)):
        y0 = rng.standard_normal(n)
        y = dev(y0.copy())
        p.level_smooth(0, dev(x), y, beta=beta, sweeps=sweeps)
        t = d * x
        for _ in range(sweeps - 1):
            t = d * (x - nd @ t)
        ref = y0 + t if beta else t
        assert np.abs(y.cpu().numpy() - ref).max() <= 1e-13 * np.abs(ref).max(), (sweeps, beta)


@pytest.mark.parametrize("idim", [33, 40, 47])
def test_dia_classes_cycle(eng, orc, idim):
    """FP64 and FP32-mixed solves on a 3-D Poisson level of this form against
    the oracle: iterations and solution."""
    a = orc.gen_pde3d(idim)
    A = a.to_scipy()
    b = np.random.default_rng(idim).uniform(-1.0, 1.0, A.shape[0])
    po = orc.Prec(orc.config1_params(smoother=100, sweeps_pre=2, sweeps_post=2)).build(a)
    xo, ito, erro = po.krylov("CG", b, eps=1e-8)
    for precision in ("double", "mixed"):
        p = eng.MldPrec(device=0).init("ML")
        for k, v in (("SMOOTHER_TYPE", "L1-JACOBI"), ("SMOOTHER_SWEEPS", 2), ("AGGR_THRESH", 0.0),
                     ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 200), ("COARSE_SOLVE", "BJAC"),
                     ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
            p.set(k, v)
        p.set_precision(precision).build(A)
        for method in ("CG", "FCG"):
            x, it, err = eng.psb_krylov(method, A, p, dev(b), eps=1e-8)
            assert err <= 1e-8 and abs(it - ito) <= 1
            assert np.abs(x.cpu().numpy() - xo).max() <= 1e-6 * np.abs(xo).max()
