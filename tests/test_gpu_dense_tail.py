"""Dense tail operators of more than 1024 rows, formed by the cycle on all
unit vectors at once: the same operator as the level-by-level cycle
(MLD_DENSE_TAIL=0) to 1e-12 (FP64, the bar of the smaller tails) and 1e-5
(FP32), for every smoother and cycle that has one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("smoother,sweeps,cycle,extra", [
    ("FBGS", 1, "VCYCLE", ()), ("FBGS", 2, "WCYCLE", ()), ("BJAC", 1, "VCYCLE", ()), ("BJAC", 1, "ADD", ()),
    ("JACOBI", 1, "ADD", ()), ("L1-JACOBI", 3, "WCYCLE", ()), ("JACOBI", 2, "VCYCLE", (("SMOOTHER_SWEEPS", 0, "PRE"),)),
    ("FBGS", 1, "ADD", ())])
@pytest.mark.parametrize("idim", [251, 301])
def test_large_tail(eng, monkeypatch, smoother, sweeps, cycle, extra, idim):
    import mld2p4_amd.problems as problems

    a = problems.pde2d_poisson(idim, single_h=False)

    def build(precision):
        p = eng.MldPrec(device=0).init("ML")
        for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", sweeps), ("ML_CYCLE", cycle),
                     ("AGGR_THRESH", 0.0), ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 100),
                     ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
            p.set(k, v)
        for k, v, pos in extra:
            p.set(k, v, pos=pos)
        return p.set_precision(precision).build(a)

    print(f"[large tail] {idim}x{idim} {smoother} {sweeps} {cycle} {extra}", flush=True)
    x = torch.from_numpy(np.random.default_rng(idim).standard_normal(idim * idim)).to("cuda:0")
    y = {}
    for precision in ("double", "mixed"):
        p = build(precision)
        lev = p.dense_tail()
        assert lev == 2 and 1024 < p.level_info(lev)["n"], [p.level_info(l)["n"] for l in range(p.nlev)]
        monkeypatch.setenv("MLD_DENSE_TAIL", "0")
        q = build(precision)
        monkeypatch.delenv("MLD_DENSE_TAIL")
        assert q.dense_tail() == -1
        yp, y[precision] = p.apply(x), q.apply(x)
        bar = 1e-12 if precision == "double" else 1e-5
        assert float((yp - y[precision]).abs().max() / y[precision].abs().max()) <= bar


@pytest.mark.parametrize("smoother,cycle,extra", [
    ("JACOBI", "VCYCLE", ()), ("L1-JACOBI", "WCYCLE", ()), ("BJAC", "VCYCLE", ()), ("BJAC", "ADD", ()),
    ("JACOBI", "ADD", (("SMOOTHER_TYPE", "BJAC", "POST"),)), ("JACOBI", "VCYCLE", (("SMOOTHER_TYPE", "BJAC", "POST"),)),
    ("JACOBI", "MULT", (("SMOOTHER_SWEEPS", 3, "PRE"), ("SMOOTHER_SWEEPS", 2, "POST")))])
@pytest.mark.parametrize("idim", [15, 70, 251])
def test_transposed_tail(eng, monkeypatch, smoother, cycle, extra, idim):
    """'T' with the tail's operator transposed, where the transposed cycle is
    that operator: as without a tail, 1e-12 in FP64 and 1e-5 in FP32, on an
    unsymmetric operator (convection)."""
    import scipy.sparse as sp

    n = idim * idim
    one = np.ones(n)
    right = np.where((np.arange(n) + 1) % idim != 0, -1.4, 0.0)
    left = np.where(np.arange(n) % idim != 0, -0.6, 0.0)
    a = sp.diags([-one[idim:], left[1:], 4.3 * one, right[:-1], -0.8 * one[idim:]], [-idim, -1, 0, 1, idim],
                 format="csr")

    def build(precision):
        p = eng.MldPrec(device=0).init("ML")
        for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", 2 if smoother != "BJAC" else 1),
                     ("ML_CYCLE", cycle), ("AGGR_THRESH", 0.0), ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 20),
                     ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 1)):
            p.set(k, v)
        for k, v, pos in extra:
            p.set(k, v, pos=pos)
        return p.set_precision(precision).build(a)

    print(f"[transposed tail] {idim}x{idim} {smoother} {cycle} {extra}", flush=True)
    x = torch.from_numpy(np.random.default_rng(idim).standard_normal(n)).to("cuda:0")
    for precision in ("double", "mixed"):
        p = build(precision)
        assert p.dense_tail() >= 1
        monkeypatch.setenv("MLD_DENSE_TAIL", "0")
        q = build(precision)
        monkeypatch.delenv("MLD_DENSE_TAIL")
        yq = q.apply(x, trans="T")
        for _ in range(2):
            yp = p.apply(x, trans="T")
            bar = 1e-12 if precision == "double" else 1e-5
            assert float((yp - yq).abs().max() / yq.abs().max()) <= bar
        yn, ym = p.apply(x), q.apply(x)
        assert float((yn - ym).abs().max() / ym.abs().max()) <= bar


@pytest.mark.parametrize("cycle", ["KCYCLE", "KCYCLESYM"])
@pytest.mark.parametrize("idim,mcs", [(9, 40), (24, 40), (24, 500), (33, 2000)])
def test_kcycle_coarsest(eng, orc, monkeypatch, cycle, idim, mcs):
    """Below a K-cycle the coarsest level's ILU(0) solver as one product: as
    without, for solves and applications; dense_tail() names no level."""
    print(f"[K-cycle coarsest] {cycle} {idim} {mcs}", flush=True)
    A = orc.gen_pde3d(idim).to_scipy()
    x = torch.from_numpy(np.random.default_rng(idim).standard_normal(A.shape[0])).to("cuda:0")
    for precision, bar in (("double", 1e-11), ("mixed", 1e-4)):
        y, z = [], []
        for off in (False, True):
            if off:
                monkeypatch.setenv("MLD_DENSE_TAIL", "0")
            p = eng.MldPrec(device=0).init("ML")
            for k, v in (("SMOOTHER_TYPE", "L1-JACOBI"), ("ML_CYCLE", cycle), ("AGGR_THRESH", 0.0),
                         ("MIN_COARSE_SIZE", mcs), ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU")):
                p.set(k, v)
            p.set_precision(precision).build(A)
            monkeypatch.delenv("MLD_DENSE_TAIL", raising=False)
            assert p.dense_tail() == -1
            y.append(p.apply(x))
            z.append(eng.psb_krylov("FCG", A, p, x, eps=1e-8))
        assert float((y[0] - y[1]).abs().max() / y[1].abs().max()) <= bar
        assert z[0][1] == z[1][1]
        assert float((z[0][0] - z[1][0]).abs().max() / z[1][0].abs().max()) <= 1e-6
