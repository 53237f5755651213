"""Forms that products can do without (row classes, value tables, packed
factors, dense tails and their transposes) are left out where there is no room
for them: the hierarchy is built and solves as before, level by level and from
the stored arrays."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def build(eng, A, smoother, cycle, precision):
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", smoother), ("SMOOTHER_SWEEPS", 2 if "JACOBI" in smoother else 1),
                 ("ML_CYCLE", cycle), ("AGGR_THRESH", 0.0), ("AGGR_PROL", "SMOOTHED"), ("MIN_COARSE_SIZE", 100),
                 ("COARSE_SOLVE", "BJAC"), ("COARSE_SUBSOLVE", "ILU"), ("COARSE_SWEEPS", 4)):
        p.set(k, v)
    return p.set_precision(precision).build(A)


@pytest.mark.parametrize("smoother,cycle,precision", [
    ("L1-JACOBI", "VCYCLE", "double"), ("L1-JACOBI", "VCYCLE", "mixed"), ("BJAC", "VCYCLE", "double"),
    ("L1-JACOBI", "KCYCLESYM", "double")])
def test_left_out(eng, orc, monkeypatch, capfd, smoother, cycle, precision):
    print(f"[optional room] {smoother} {cycle} {precision}", flush=True)
    idim = 72
    A = orc.gen_pde3d(idim).to_scipy()
    b = np.random.default_rng(idim).standard_normal(A.shape[0])
    bd = torch.from_numpy(b).to("cuda:0")
    monkeypatch.setenv("MLD_VERBOSE", "1")
    monkeypatch.setenv("MLD_AUTOTUNE", "0")  # the same layouts in every build, so that their memory can be compared
    its, held = {}, {}
    for room in ("0", "1", "20", None):
        if room is None:
            monkeypatch.delenv("MLD_EXTRA_MB")
        else:
            monkeypatch.setenv("MLD_EXTRA_MB", room)
        capfd.readouterr()
        p = build(eng, A, smoother, cycle, precision)
        err = capfd.readouterr().err
        # A and ND of the fine level (class bytes) and the dense tail: over 1 MB each here, packed factors over 20
        forms = [p.op_bytes_form(0, "A") == "DIA+rows", "packed for one workgroup" in err and "44723-row" in err]
        if room == "0":
            assert not any(forms) and p.dense_tail() == -1 and "distinct" not in err
        if room is None:
            assert forms[0] and (smoother != "BJAC" or forms[1])
            assert (p.dense_tail() > 0) == (cycle == "VCYCLE")
        if room in ("0", "1", "20"):
            assert not forms[1]
        held[room] = p.device_bytes()
        x, it, e = eng.psb_krylov("FCG", A, p, bd, eps=1e-8)
        assert e <= 1e-8 and np.linalg.norm(b - A @ x.cpu().numpy()) <= 1.01e-8 * np.linalg.norm(b)
        its[room] = it
        x, it, e = eng.psb_krylov_adjoint("CG", p, bd, eps=1e-8)
        assert e <= 1e-8 and np.linalg.norm(b - A.T @ x.cpu().numpy()) <= 1.01e-8 * np.linalg.norm(b)
    assert max(its.values()) - min(its.values()) <= 1
    assert held["0"] <= held["1"] <= held["0"] + 1e6 and held["20"] <= held["0"] + 20e6 and held["0"] < held[None]
