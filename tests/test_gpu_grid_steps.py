"""Grid substitutions take their steps (grid lines + 14) in batches of 8, two
in turn: the sequential ones' values bit for bit at step counts around whole
batches, in both directions, with ILU(0) and Gauss-Seidel."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("smoother", ["BJAC", "FBGS"])
@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("idim", [26, 27, 33, 34, 35, 42, 63])
def test_batches(eng, orc, monkeypatch, smoother, precision, idim):
    print(f"[grid steps] {smoother} {precision} {idim}", flush=True)
    A = orc.gen_pde3d(idim).to_scipy()
    x = torch.from_numpy(np.random.default_rng(idim).standard_normal(A.shape[0])).to("cuda:0")
    y = []
    monkeypatch.setenv("MLD_AUTOTUNE", "0")  # both handles' products in the same layouts, not the faster ones of two timings
    for off in (False, True):
        if off:
            monkeypatch.setenv("MLD_TRSV_GRID", "0")
        p = eng.MldPrec(device=0).init("ML")
        for k, v in (("SMOOTHER_TYPE", smoother), ("AGGR_THRESH", 0.0), ("MIN_COARSE_SIZE", 200),
                     ("SUB_SOLVE", "ILU"), ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU")):
            if k != "SUB_SOLVE" or smoother == "BJAC":
                p.set(k, v)
        p.set_precision(precision).build(A)
        y.append([p.apply(x) for _ in range(2)])
    monkeypatch.delenv("MLD_TRSV_GRID")
    for a in y[0] + y[1][1:]:
        assert torch.equal(a, y[1][0])
