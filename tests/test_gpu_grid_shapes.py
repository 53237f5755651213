"""Grid substitutions on boxes whose sides differ, with unequal coefficients
(an exchanged side or stride shows): both solves of ILU(0) and Gauss-Seidel
bit for bit as the sequential ones, the grid form read back."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def box(nx, ny, nz, seed):
    """7-point matrix on an nx x ny x nz grid (x fastest), every coefficient its own."""
    n = nx * ny * nz
    rng = np.random.default_rng(seed)
    i = np.arange(n)
    x, y, z = i % nx, i // nx % ny, i // (nx * ny)
    rows, cols, vals = [], [], []
    for o, ok in ((-nx * ny, z > 0), (-nx, y > 0), (-1, x > 0), (1, x < nx - 1), (nx, y < ny - 1),
                  (nx * ny, z < nz - 1)):
        rows.append(i[ok])
        cols.append(i[ok] + o)
        vals.append(-rng.uniform(0.5, 1.5, ok.sum()))
    a = sp.csr_matrix((np.concatenate(vals), (np.concatenate(rows), np.concatenate(cols))), shape=(n, n))
    a = (a + sp.diags(np.asarray(abs(a).sum(axis=1)).ravel() + 0.1)).tocsr()
    a.sort_indices()
    return a


@pytest.mark.parametrize("smoother", ["BJAC", "FBGS"])
@pytest.mark.parametrize("nx,ny,nz", [(17, 40, 31), (64, 25, 33), (9, 64, 47), (2, 130, 33), (101, 26, 32),
                                      (33, 121, 9)])
def test_boxes(eng, orc, monkeypatch, capfd, smoother, nx, ny, nz):
    print(f"[grid shapes] {smoother} {nx} x {ny} x {nz}", flush=True)
    A = box(nx, ny, nz, nx + ny + nz)
    monkeypatch.setenv("MLD_VERBOSE", "1")
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", 1), ("AGGR_THRESH", 0.0), ("AGGR_PROL", "SMOOTHED"),
                 ("MIN_COARSE_SIZE", 40), ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
        p.set(k, v)
    capfd.readouterr()
    p.build(A)
    assert f"on a {nx} x {ny} x {nz} grid: grid substitutions" in capfd.readouterr().err
    po = orc.Prec(orc.config1_params(smoother={"BJAC": 2, "FBGS": 4}[smoother], min_coarse_size=40))
    po = po.build(orc.Csr.from_scipy(A))
    n = A.shape[0]
    rng = np.random.default_rng(n)
    for which in ((0, 1) if smoother == "FBGS" else (0,)):
        for beta in (0, 1, 0):
            x, y0 = rng.standard_normal(n), rng.standard_normal(n)
            y = torch.from_numpy(y0.copy()).to("cuda:0")
            p.level_smooth(0, torch.from_numpy(x).to("cuda:0"), y, beta=beta, sweeps=1, which=which)
            yo = po.smooth(0, x, alpha=1.0, beta=float(beta), y=y0, sweeps=1, which=which)
            assert (y.cpu().numpy() == yo).all(), (which, beta)
