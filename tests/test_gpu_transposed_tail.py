"""Which transposed cycles take the transposed dense tail operator: the ones
that are that operator, read back from the build's messages; an additive cycle
with two smoothers, which is not, keeps its level-by-level form.  Non-finite
right-hand sides stay non-finite through a tail of more than 1024 rows."""
import re

import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def convection(idim):
    n = idim * idim
    one = np.ones(n)
    right = np.where((np.arange(n) + 1) % idim != 0, -1.4, 0.0)
    left = np.where(np.arange(n) % idim != 0, -0.6, 0.0)
    return sp.diags([-one[idim:], left[1:], 4.3 * one, right[:-1], -0.8 * one[idim:]], [-idim, -1, 0, 1, idim],
                    format="csr")


def build(eng, a, smoother, cycle, extra, precision):
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", 2 if smoother != "BJAC" else 1),
                 ("ML_CYCLE", cycle), ("AGGR_THRESH", 0.0), ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 20),
                 ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 1)):
        p.set(k, v)
    for k, v, pos in extra:
        p.set(k, v, pos=pos)
    return p.set_precision(precision).build(a)


@pytest.mark.parametrize("smoother,cycle,extra,used", [
    ("JACOBI", "VCYCLE", (), True), ("L1-JACOBI", "WCYCLE", (), True), ("BJAC", "VCYCLE", (), True),
    ("BJAC", "ADD", (), True), ("JACOBI", "VCYCLE", (("SMOOTHER_TYPE", "BJAC", "POST"),), True),
    ("JACOBI", "ADD", (("SMOOTHER_TYPE", "BJAC", "POST"),), False)])
@pytest.mark.parametrize("idim", [70, 251])
def test_taken(eng, monkeypatch, capfd, smoother, cycle, extra, used, idim):
    print(f"[transposed tail taken] {idim} {smoother} {cycle}", flush=True)
    a = convection(idim)
    x = torch.from_numpy(np.random.default_rng(idim).standard_normal(idim * idim)).to("cuda:0")
    monkeypatch.setenv("MLD_VERBOSE", "1")
    for precision in ("double", "mixed"):
        p = build(eng, a, smoother, cycle, extra, precision)
        assert p.dense_tail() >= 1
        capfd.readouterr()
        p.apply(x, trans="T")
        lines = re.findall(r"transposed dense tail of (\d+) rows: off by (\S+) of its largest value, (\w+)",
                           capfd.readouterr().err)
        assert len(lines) == 1 and int(lines[0][0]) == p.level_info(p.dense_tail())["n"]
        assert (lines[0][2] == "used") == used, (precision, lines)


@pytest.mark.parametrize("smoother", ["L1-JACOBI", "BJAC"])
def test_not_finite(eng, monkeypatch, smoother):
    a = convection(251)
    n = a.shape[0]
    for value in (np.inf, -np.inf, np.nan):
        x = np.random.default_rng(1).standard_normal(n)
        x[n // 3] = value
        y = []
        for off in (False, True):
            if off:
                monkeypatch.setenv("MLD_DENSE_TAIL", "0")
            p = build(eng, a, smoother, "VCYCLE", (), "double")
            monkeypatch.delenv("MLD_DENSE_TAIL", raising=False)
            assert off or p.level_info(p.dense_tail())["n"] > 1024
            y.append(p.apply(torch.from_numpy(x).to("cuda:0")).cpu().numpy())
        bad = [~np.isfinite(v) for v in y]
        assert bad[1].any() and bad[0][bad[1]].all()
