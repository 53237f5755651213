"""Dot products of the Krylov loop, added by the block that ends last on small
systems and by a kernel of their own on large ones: CG residuals at sizes
around one block, one group of blocks and the least size of the second form.
The sums are in a fixed order, so that every solve gives the same bits, and a
solve leaves the counters of the next at zero."""
import numpy as np
import pytest
import scipy.sparse as sp

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

EDGE = 2048 * 512  # blocks that add their own sums times rows per block


@pytest.mark.parametrize("n", [1, 2, 255, 511, 512, 513, 1025, 32 * 512 - 1, 32 * 512 + 1, 33 * 512,
                               100003, EDGE - 1, EDGE, EDGE + 1, EDGE + 513])
@pytest.mark.parametrize("method", ["CG", "FCG"])
def test_dots(eng, n, method):
    """Five iterations against the same recurrence in numpy: a sum of n
    products rounded in another order differs by a few n^0.5 eps of its
    value, and five steps of a system of condition <= 3 do not amplify it
    beyond 1e3 of that: 1e-10 at 10^6 rows."""
    print(f"[dots] n {n} {method}", flush=True)
    rng = np.random.default_rng(n)
    d = rng.uniform(4.0, 6.0, n)
    off = np.full(max(n - 1, 0), -1.0)
    A = sp.diags([off, d, off], [-1, 0, 1], format="csr") if n > 1 else sp.csr_matrix([[d[0]]])
    b = rng.standard_normal(n)
    prec = eng.MldPrec(device=0).init("JACOBI").build(A)
    x, it, err = eng.psb_krylov(method, A, prec, torch.from_numpy(b).to("cuda:0"), eps=1e-30, itmax=5)
    xs = [eng.psb_krylov(method, A, prec, torch.from_numpy(b).to("cuda:0"), eps=1e-30, itmax=5)[0] for _ in range(3)]
    for y in xs:
        assert torch.equal(x, y)
    xr, r = np.zeros(n), b.copy()
    rho = p = None
    for _ in range(it):
        z = r / d
        new = r @ z
        if new == 0.0:
            break
        p = z if p is None else z + (new / rho) * p
        q = A @ p
        al = new / (p @ q)
        xr += al * p
        r = r - al * q
        rho = new
    assert np.abs(x.cpu().numpy() - xr).max() <= 1e-10 * np.abs(xr).max()
    if n > 16:  # below, the residual is all rounding before the fifth step
        assert it == 5 and abs(err - np.linalg.norm(r) / np.linalg.norm(b)) <= 1e-10


@pytest.mark.parametrize("method", ["CG", "FCG"])
@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("idim,eps", [(5, 1e-3), (12, 1e-6), (24, 1e-8), (24, 1e-2)])
def test_ahead(eng, orc, idim, eps, precision, method):
    """A cycle enqueued before the residual norm is known changes nothing: a
    solve that stops by its tolerance, by the same number of iterations, and
    again after both, gives the same bits."""
    print(f"[ahead] {idim} {eps} {precision} {method}", flush=True)
    A = orc.gen_pde3d(idim).to_scipy()
    b = torch.from_numpy(np.random.default_rng(idim).uniform(-1.0, 1.0, A.shape[0])).to("cuda:0")
    p = eng.MldPrec(device=0).init("ML")
    for k, v in (("SMOOTHER_TYPE", "L1-JACOBI"), ("AGGR_THRESH", 0.0), ("MIN_COARSE_SIZE", 20)):
        p.set(k, v)
    p.set_precision(precision).build(A)
    x, it, err = eng.psb_krylov(method, A, p, b, eps=eps)
    assert err <= eps
    y, jt, e2 = eng.psb_krylov(method, A, p, b, eps=1e-300, itmax=it)
    assert jt == it and e2 == err and torch.equal(x, y)
    z, kt, e3 = eng.psb_krylov(method, A, p, b, eps=eps)
    assert kt == it and e3 == err and torch.equal(x, z)
