"""Triangular substitutions of one workgroup over a packed factor (ILU and
Gauss-Seidel levels whose level sets are narrow), bit for bit against the
oracle's sequential sweeps: slices of less than, exactly and more than 64 rows
(grids with 61 to 130 lines), rows longer than the entries held in registers
(ILU(k)), the smallest levels that take this form, 1 and 2 sweeps, beta 0 and
1, repeated applications; FP32 within rounding of FP64; a right-hand side with
infinities and zeros of both signs."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def grid2d(nx, ny, nine=False):
    """5- or 9-point matrix on an nx x ny grid with unequal coefficients."""
    n = nx * ny
    rng = np.random.default_rng(nx * 1000 + ny)
    i = np.arange(n)
    x, y = i % nx, i // nx
    rows, cols, vals = [], [], []
    for dx in (-1, 0, 1):
        for dy in (-1, 0, 1):
            if (dx == 0 and dy == 0) or (not nine and dx != 0 and dy != 0):
                continue
            ok = (x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny)
            rows.append(i[ok])
            cols.append((i + dx + nx * dy)[ok])
            vals.append(-rng.uniform(0.5, 1.5, ok.sum()))
    a = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))), shape=(n, n))
    a = a + sp.diags(np.asarray(np.abs(a).sum(axis=1)).ravel() + 0.1)
    a = a.tocsr()
    a.sort_indices()
    return a


def build(eng, orc, A, smoother, precision="double", extra=(), **kw):
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", 1), ("AGGR_THRESH", 0.0),
                 ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 40), ("COARSE_SOLVE", "BJAC"),
                 ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)) + tuple(extra):
        p.set(k, v)
    p.set_precision(precision).build(A)
    po = orc.Prec(orc.config1_params(smoother={"BJAC": 2, "FBGS": 4}[smoother], min_coarse_size=40, **kw))
    return p, po.build(orc.Csr.from_scipy(A))


@pytest.mark.parametrize("nx,ny,nine", [(12, 11, False), (40, 17, True), (61, 64, False), (64, 64, False),
                                        (65, 130, False), (130, 67, True), (1500, 9, False), (211, 203, False)])
def test_gauss_seidel_packed(eng, orc, nx, ny, nine):
    A = grid2d(nx, ny, nine)
    p, po = build(eng, orc, A, "FBGS")
    for lev in range(p.nlev - 1):
        n = p.level_info(lev)["n"]
        rng = np.random.default_rng(n)
        for which, sweeps, beta in ((0, 1, 0), (1, 1, 1), (0, 2, 1), (1, 2, 0), (0, 1, 0)):
            print(f"[GS packed] {nx}x{ny} level {lev} n {n} which {which} sweeps {sweeps} beta {beta}", flush=True)
            x, y0 = rng.standard_normal(n), rng.standard_normal(n)
            y = dev(y0.copy())
            p.level_smooth(lev, dev(x), y, beta=beta, sweeps=sweeps, which=which)
            yo = po.smooth(lev, x, alpha=1.0, beta=float(beta), y=y0, sweeps=sweeps, which=which)
            assert (y.cpu().numpy() == yo).all()


@pytest.mark.parametrize("nx,ny,fill", [(12, 12, 0), (33, 30, 0), (64, 65, 1), (47, 52, 8), (40, 44, 20)])
def test_ilu_packed(eng, orc, nx, ny, fill):
    A = grid2d(nx, ny, nine=fill > 1)
    p, po = build(eng, orc, A, "BJAC", extra=(("SUB_SOLVE", "ILU"), ("SUB_FILLIN", fill)), sub_fill=fill)
    for lev in range(p.nlev - 1):
        n = p.level_info(lev)["n"]
        rng = np.random.default_rng(n + fill)
        for beta in (0, 1, 0):
            print(f"[ILU packed] {nx}x{ny} fill {fill} level {lev} n {n} beta {beta} "
                  f"longest row {np.diff(p.level_csr(lev, 'L').indptr).max()}", flush=True)
            x, y0 = rng.standard_normal(n), rng.standard_normal(n)
            y = dev(y0.copy())
            p.level_smooth(lev, dev(x), y, beta=beta, sweeps=1)
            yo = po.smooth(lev, x, alpha=1.0, beta=float(beta), y=y0, sweeps=1)
            assert (y.cpu().numpy() == yo).all()


def test_packed_special_values(eng, orc):
    """Infinities and zeros of both signs in the right-hand side travel as in
    the sequential sweep (padding entries add nothing)."""
    A = grid2d(70, 66)
    p, po = build(eng, orc, A, "FBGS")
    n = A.shape[0]
    x = np.random.default_rng(9).standard_normal(n)
    x[::7] = 0.0
    x[::11] = -0.0
    x[n - 3] = np.inf
    y = dev(np.zeros(n))
    p.level_smooth(0, dev(x), y)
    yo = po.smooth(0, x, alpha=1.0, beta=0.0, y=np.zeros(n), sweeps=1)
    yg = y.cpu().numpy()
    assert np.array_equal(yg, yo, equal_nan=True) and np.array_equal(np.signbit(yg), np.signbit(yo))


def test_packed_fp32(eng, orc):
    """FP32 hierarchy: the preconditioned vector within FP32 rounding of the
    oracle's FP64 one (the bar of the other FP32 applications, 1e-5)."""
    A = grid2d(130, 67)
    for sm in ("FBGS", "BJAC"):
        p, po = build(eng, orc, A, sm, precision="mixed")
        x = np.random.default_rng(4).standard_normal(A.shape[0])
        y = p.apply(dev(x)).cpu().numpy()
        yo = po.apply(x)
        assert np.abs(y - yo).max() <= 1e-5 * np.abs(yo).max()
