"""How often a solve applies the preconditioner: exactly once per iteration
where enqueuing the next application early would gain nothing (triangular
solves on the fine level, more than 2^21 rows, K-cycles), at most once more
elsewhere; twice per iteration at most in BiCGStab."""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("smoother,sweeps,cycle,idim,spare", [
    ("FBGS", 1, "VCYCLE", 96, 0), ("BJAC", 1, "VCYCLE", 40, 0), ("FBGS", 1, "VCYCLE", 33, 0),
    ("L1-JACOBI", 2, "VCYCLE", 136, 0), ("L1-JACOBI", 2, "KCYCLESYM", 40, 0),
    ("JACOBI", 1, "VCYCLE", 40, 1), ("L1-JACOBI", 2, "VCYCLE", 48, 1)])
def test_counts(eng, orc, monkeypatch, capfd, smoother, sweeps, cycle, idim, spare):
    print(f"[applications] {smoother} {cycle} {idim}", flush=True)
    A = orc.gen_pde3d(idim).to_scipy()
    b = torch.from_numpy(np.random.default_rng(idim ** 3).uniform(-1.0, 1.0, idim ** 3)).to("cuda:0")
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", sweeps), ("ML_CYCLE", cycle), ("AGGR_THRESH", 0.0),
                 ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 200), ("COARSE_SOLVE", "BJAC"),
                 ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
        p.set(k, v)
    p.build(A)
    monkeypatch.setenv("MLD_VERBOSE", "1")
    for method in ("CG", "FCG", "BICGSTAB"):
        for eps in (1e-6, 3e-7, 1e-7, 1e-8, 1e-9):
            capfd.readouterr()
            x, it, err = eng.psb_krylov(method, A, p, b, eps=eps)
            lines = re.findall(r"solve of (\d+) rows: (\d+) iterations, (\d+) applications", capfd.readouterr().err)
            assert err <= eps and len(lines) == 1
            rows, its, app = (int(q) for q in lines[0])
            assert rows == idim ** 3 and its == it
            if method == "BICGSTAB":
                assert 2 * it - 1 <= app <= 2 * it
            else:
                assert it <= app <= it + spare, (method, eps)
