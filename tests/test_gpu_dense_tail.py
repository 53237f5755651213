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
