"""Block solves whose solution updates lag one iteration behind, and block
products of the small levels with one workgroup per row: every column as the
single-vector solver stopped after the same number of iterations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).to("cuda:0")


def build(eng, A, precision, mcs):
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", "L1-JACOBI"), ("SMOOTHER_SWEEPS", 2), ("AGGR_THRESH", 0.0),
                 ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", mcs), ("COARSE_SOLVE", "BJAC"),
                 ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
        p.set(k, v)
    return p.set_precision(precision).build(A)


@pytest.mark.parametrize("method", ["CG", "FCG"])
@pytest.mark.parametrize("precision,tol", [("double", 1e-10), ("mixed", 1e-4)])
@pytest.mark.parametrize("idim,mcs", [(9, 20), (17, 40), (24, 200)])
def test_steps(eng, orc, method, precision, tol, idim, mcs):
    """Iterates, not only limits: itmax 0 to 6, a zero column, a column that
    starts at its solution and one that converges early.  Two orders of
    summation in the cycle differ by its rounding (1e-13 FP64, 1e-6 FP32),
    which a few steps amplify by at most the cycle's condition (< 100)."""
    print(f"[block steps] {method} {precision} {idim}", flush=True)
    A = orc.gen_pde3d(idim).to_scipy()
    n = A.shape[0]
    p = build(eng, A, precision, mcs)
    rng = np.random.default_rng(idim)
    B = rng.standard_normal((32, n))
    X0 = rng.standard_normal((32, n))
    B[3] = 0.0
    X0[3] = 0.0
    B[8] = A @ X0[8]
    B[21] = A @ X0[21] + 1e-7 * B[21]
    for itmax in (0, 1, 2, 6):
        X, it, er = p.krylov_block(method, dev(B), X=dev(X0.copy()), eps=1e-8, itmax=itmax)
        X = X.cpu().numpy()
        assert it.max() <= itmax and it[3] == 0 and it[8] == 0
        assert (X[3] == 0).all() and (X[8] == X0[8]).all()
        for j in (0, 5, 21, 31):
            x, _, _ = eng.psb_krylov(method, A, p, dev(B[j]), x=dev(X0[j].copy()), eps=1e-300, itmax=int(it[j]))
            x = x.cpu().numpy()
            assert np.abs(X[j] - x).max() <= tol * np.abs(x).max(), (itmax, j)


@pytest.mark.parametrize("precision,tol", [("double", 1e-12), ("mixed", 1e-5)])
@pytest.mark.parametrize("idim,mcs", [(8, 30), (20, 40), (30, 100), (33, 3000)])
def test_long_rows(eng, orc, precision, tol, idim, mcs):
    """Levels below 4096 rows with 16 and more entries per row (rows of fewer
    and of more than 32, 128 entries), against the oracle's cycle."""
    print(f"[long rows] {precision} {idim} {mcs}", flush=True)
    a = orc.gen_pde3d(idim)
    A = a.to_scipy()
    p = build(eng, A, precision, mcs)
    po = orc.Prec(orc.config1_params(smoother=orc.SM_L1JAC, sweeps_pre=2, sweeps_post=2, min_coarse_size=mcs)).build(a)
    X = np.random.default_rng(idim).standard_normal((32, A.shape[0]))
    Y = p.apply_block(dev(X)).cpu().numpy()
    for j in (0, 13, 31):
        yo = po.apply(X[j])
        assert np.abs(Y[j] - yo).max() <= tol * np.abs(yo).max(), j
