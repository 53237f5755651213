"""Packed forms (row classes, value tables) of a Jacobi level's operators: of
those that its sweeps read and of no other; the same results with every number
of sweeps."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("fmt", ["auto", "sell"])
@pytest.mark.parametrize("sweeps", [1, 2, 3])
def test_forms_and_results(eng, orc, monkeypatch, capfd, fmt, sweeps):
    print(f"[packed forms] {fmt} {sweeps}", flush=True)
    idim = 64
    A = orc.gen_pde3d(idim).to_scipy()
    n = A.shape[0]
    monkeypatch.setenv("MLD_VERBOSE", "1")
    p = eng.MldPrec(device=0).init("JACOBI")
    p.set("SMOOTHER_SWEEPS", sweeps)
    p.set_format(fmt)
    capfd.readouterr()
    p.build(A)
    err = capfd.readouterr().err
    assert sum("distinct" in q for q in err.splitlines()) == sweeps  # A; ND D from two sweeps on; ND from three
    x = np.random.default_rng(sweeps).standard_normal(n)
    d = 1.0 / A.diagonal()
    nd = (A - sp.diags(A.diagonal())).tocsr()
    for k in (1, 2, 3, 4):  # also numbers of sweeps that the level does not have
        y = torch.zeros(n, dtype=torch.float64, device="cuda:0")
        p.level_smooth(0, torch.from_numpy(x).to("cuda:0"), y, sweeps=k)
        t = d * x
        for _ in range(k - 1):
            t = d * (x - nd @ t)
        assert np.abs(y.cpu().numpy() - t).max() <= 1e-13 * np.abs(t).max(), k
